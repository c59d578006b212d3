"""The projection guess at every window of its Gram kernel (1 to 6 signals together, windows of 4 with a
remainder beyond), row counts around its tiles: the solutions of the quadratic extrapolation, in fewer
iterations."""
import numpy as np
import pytest

import dmri_mesh as dm
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("per_gdir", [False, True])
@pytest.mark.parametrize("nsig", [1, 2, 3, 4, 5, 6, 7, 9, 64])
@pytest.mark.parametrize("nv", [90, 1300])
def test_projection_matches_extrapolation(nsig, per_gdir, nv):
    import dmri_native as N

    m = dm.cylinder_mesh(5.0, 5.0, nv, seed=2)
    fA, fB = O.gcloud_sequence(O.pgse_piecewise(3000.0, 4000.0), 7000.0, 200.0)
    qs = np.array([O.q_from_b_pgse(b, 10600.0, 43100.0) for b in np.linspace(500.0, 4000.0, nsig)])
    gd = np.random.default_rng(1).normal(size=(nsig, 3)) if per_gdir else (0.0, 1.0, 0.0)
    ctx = N.Context(0)
    ctx.set_mesh(m.xyz, m.tets)
    ctx.set_coeffs(D=3e-3)
    ctx.assemble()
    a, sa = ctx.solve_batched(fA, fB, 200.0, qs, gd, rtol=1e-13, krylov="cocg")
    b, sb = ctx.solve_batched(fA, fB, 200.0, qs, gd, rtol=1e-13, krylov="cocg", guess=3)
    assert np.max(np.abs(a - b) / np.abs(b)) <= 1e-11
    assert sa["iters_total"] < sb["iters_total"]
