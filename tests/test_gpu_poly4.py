"""The degree-4 polynomial of the real part: the solutions of plain Jacobi, in under half of its products
with the operator (three quarters for mild steps), for every Krylov method, on both sides of the size it starts at, over one-lane staged rows and rows
on several lanes, one direction and several, stiff and mild steps, with the FP32 input."""
import numpy as np
import pytest

import dmri_mesh as dm
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("krylov,nsig,nv,dt,opts", [
    ("bicgstab", 1, 45000, 200.0, {}), ("bicgstab", 5, 9000, 2000.0, {}), ("bicgstab", 16, 3000, 200.0, {}),
    ("cocg", 1, 45000, 2000.0, {}), ("cocg", 1, 45000, 20.0, {}), ("cocg", 3, 700, 400.0, {}),
    ("cocg", 5, 9000, 400.0, dict(pre_fp32=1)), ("cocg", 2, 9000, 400.0, dict(mapping=1, lanes=16)),
    ("cocg", 33, 2000, 400.0, {}), ("gmres", 1, 3000, 2000.0, {}), ("gmres", 7, 700, 400.0, {})])
@pytest.mark.parametrize("per_gdir", [False, True])
def test_degree_four_matches_jacobi(krylov, nsig, nv, dt, opts, per_gdir):
    import dmri_native as N

    if per_gdir and nsig == 1:
        pytest.skip("one signal has one direction")
    m = dm.cylinder_mesh(6.0, 6.0, nv, seed=8, interface_radii=(3.0,))
    fA, fB = O.gcloud_sequence(O.pgse_piecewise(3 * dt, 4 * dt), 7 * dt, dt)
    # a gradient weak enough for the polynomial of the real part
    qs = np.linspace(0.3, 1.0, nsig) * 2e-5 * 400.0 / dt
    gd = np.random.default_rng(2).normal(size=(nsig, 3)) if per_gdir else (0.2, 1.0, 0.1)
    ctx = N.Context(0)
    ctx.set_mesh(m.xyz, m.tets, m.phase)
    ctx.set_coeffs(D=3e-3, kappa=1e-5)
    ctx.assemble()
    a, st = ctx.solve_batched(fA, fB, dt, qs, gd, rtol=1e-13, krylov=krylov, guess=1, **opts)
    ua = ctx.solution(nsig - 1)
    b, sj = ctx.solve_batched(fA, fB, dt, qs, gd, rtol=1e-13, krylov="bicgstab", precond=1, guess=1)
    assert st["precond_used"] == 2 and st["relres_max"] <= 1e-13
    assert np.max(np.abs(a - b)) <= 1e-11
    ub = ctx.solution(nsig - 1)
    assert np.linalg.norm(ua - ub) <= 1e-10 * np.linalg.norm(ub)
    # BiCGStab takes two products with the operator an iteration, the others one
    per = 2 if krylov == "bicgstab" else 1
    assert per * st["iters_total"] < (0.75 if dt < 100 else 0.5) * 2 * sj["iters_total"]
