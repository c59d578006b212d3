"""GMRES at the edges of its dot-product chunks (4 basis vectors), restart lengths 1 and 64, one signal
and as many as a launch group takes."""
import numpy as np
import pytest

import dmri_mesh as dm
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nsig,nv,restart", [(1, 130, 1), (1, 2500, 4), (1, 2500, 5), (2, 700, 8), (33, 300, 9),
                                             (64, 700, 3), (63, 130, 64), (1, 9000, 64)])
def test_gmres_matches_oracle(nsig, nv, restart):
    import dmri_native as N

    m = dm.cylinder_mesh(4.0, 4.0, nv, seed=11, interface_radii=(2.0,))
    fA, fB = O.gcloud_sequence(O.pgse_piecewise(800.0, 1200.0), 2000.0, 400.0)
    qs = np.array([O.q_from_b_pgse(b, 10600.0, 43100.0) for b in np.linspace(200.0, 4000.0, nsig)])
    ctx = N.Context(0)
    ctx.set_mesh(m.xyz, m.tets, m.phase)
    ctx.set_coeffs(D=3e-3, kappa=1e-5)
    ctx.assemble()
    sig, st = ctx.solve_batched(fA, fB, 400.0, qs, (0.0, 1.0, 0.0), rtol=1e-12, krylov="gmres", restart=restart)
    assert st["relres_max"] <= 1e-12
    S = O.System(m.xyz, m.tets, m.phase, D=3e-3, invT2=1e-16, kappa=1e-5)
    for j in sorted({0, nsig - 1}):
        ref, _, _ = S.solve((0.0, 1.0, 0.0), qs[j], 400.0, fA, fB, rtol=1e-13)
        assert abs(sig[j].real - ref) <= 1e-9 * abs(ref), (j, sig[j], ref)
