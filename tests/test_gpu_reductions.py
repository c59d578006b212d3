"""Per-signal reductions at the edges of their thread split: one signal (a column's rows over a whole
wave), counts that leave threads of a block idle, 64 signals (one thread per column), a single block of
partials and several."""
import numpy as np
import pytest

import dmri_mesh as dm
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("krylov", ["bicgstab", "cocg"])
@pytest.mark.parametrize("nsig,nv", [(1, 130), (1, 2500), (2, 700), (3, 700), (5, 2500), (7, 130), (33, 700), (63, 300),
                                     (64, 700)])
def test_batch_of_any_size_matches_oracle(nsig, nv, krylov):
    import dmri_native as N

    m = dm.cylinder_mesh(4.0, 4.0, nv, seed=11, interface_radii=(2.0,))
    fA, fB = O.gcloud_sequence(O.pgse_piecewise(800.0, 1200.0), 2000.0, 400.0)
    qs = np.array([O.q_from_b_pgse(b, 10600.0, 43100.0) for b in np.linspace(200.0, 4000.0, nsig)])
    ctx = N.Context(0)
    ctx.set_mesh(m.xyz, m.tets, m.phase)
    ctx.set_coeffs(D=3e-3, kappa=1e-5)
    ctx.assemble()
    sig, _ = ctx.solve_batched(fA, fB, 400.0, qs, (0.0, 1.0, 0.0), rtol=1e-13, krylov=krylov)
    S = O.System(m.xyz, m.tets, m.phase, D=3e-3, invT2=1e-16, kappa=1e-5)
    for j in sorted({0, nsig // 2, nsig - 1}):
        ref, _, _ = S.solve((0.0, 1.0, 0.0), qs[j], 400.0, fA, fB, rtol=1e-13)
        assert abs(sig[j].real - ref) <= 1e-9 * abs(ref), (j, sig[j], ref)
