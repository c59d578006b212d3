"""BiCGStab with its vector passes folded into the preconditioner SpMVs: the same bits as the kernels of
their own (which timed iterations keep), at sizes on both sides of the rule, with restarts off and on the
edge of the row tiles, one signal and several."""
import numpy as np
import pytest

import dmri_mesh as dm
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nsig,nv,precond", [(1, 60, 0), (1, 1000, 0), (2, 4000, 0), (5, 3000, 0), (1, 41000, 0), (3, 700, 2)])
def test_folded_iterations_equal_the_timed_ones(nsig, nv, precond):
    import dmri_native as N

    m = dm.cylinder_mesh(6.0, 6.0, nv, seed=3, interface_radii=(3.0,))
    fA, fB = O.gcloud_sequence(O.pgse_piecewise(600.0, 1000.0), 1600.0, 200.0)
    qs = np.array([O.q_from_b_pgse(b, 10600.0, 43100.0) for b in np.linspace(1000.0, 4000.0, nsig)])
    ctx = N.Context(0)
    ctx.set_mesh(m.xyz, m.tets, m.phase)
    ctx.set_coeffs(D=3e-3, kappa=1e-5)
    ctx.assemble()
    args = (fA, fB, 200.0, qs, (0.0, 1.0, 0.0))
    a, st = ctx.solve_batched(*args, rtol=1e-12, precond=precond)
    ua = ctx.solution(nsig - 1)
    b, stb = ctx.solve_batched(*args, rtol=1e-12, precond=precond, profile=3)  # the first 3 iterations timed
    ub = ctx.solution(nsig - 1)
    assert stb["kern_launches"][0] > 0 and st["iters_total"] == stb["iters_total"]
    assert np.array_equal(a, b) and np.array_equal(ua, ub)
    ref, _, _ = O.System(m.xyz, m.tets, m.phase, D=3e-3, invT2=1e-16, kappa=1e-5).solve((0.0, 1.0, 0.0), qs[0], 200.0,
                                                                                      fA, fB, rtol=1e-13)
    assert abs(a[0].real - ref) <= 1e-9 * abs(ref)
