"""The iterate a solve returns when a loose tolerance stops it: its own residual, formed on the host with the
oracle's matrices and the solver's scaling, meets that tolerance.  A solve that left out its last update returns
the iterate before, whose residual does not.  One theta step from u = 1, tolerances at fractions of the start's
residual, for every way the solver ends an iteration: folded and separate updates, degree 1 and 4, FP32 input,
one signal and groups, one direction and several."""
import numpy as np
import pytest
import scipy.sparse as sp

import dmri_mesh as dm
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("krylov,nsig,nv,dt,q,form,opts", [
    ("cocg", 1, 130, 200.0, 1.6e-4, 0, {}), ("cocg", 1, 2500, 200.0, 1.6e-4, 0, {}), ("cocg", 1, 20000, 200.0, 1e-4, 0, {}),
    ("cocg", 1, 45000, 2000.0, 4e-6, 2, {}), ("cocg", 1, 400000, 400.0, 2e-5, 2, {}),
    ("cocg", 3, 9000, 400.0, 2e-5, 2, {}), ("cocg", 2, 9000, 400.0, 2e-5, 2, dict(pre_fp32=1)),
    ("cocg", -3, 2000, 200.0, 1.6e-4, 0, {}), ("cocg", -4, 9000, 400.0, 2e-5, 2, {}),
    ("bicgstab", 1, 1000, 200.0, 1.6e-4, 0, {}), ("bicgstab", 1, 45000, 400.0, 2e-5, 2, {}),
    ("bicgstab", 3, 15000, 2000.0, 4e-6, 2, {}), ("bicgstab", 20, 1000, 200.0, 2e-5, 0, {}),
    ("bicgstab", -3, 2000, 200.0, 1.6e-4, 0, {}), ("gmres", 2, 3000, 400.0, 2e-5, 2, {})])
def test_returned_iterate_meets_the_tolerance(krylov, nsig, nv, dt, q, form, opts):
    import dmri_native as N

    per_gdir, nsig = nsig < 0, abs(nsig)
    m = dm.cylinder_mesh(6.0, 6.0, nv, seed=4, interface_radii=(3.0,))
    S = O.System(m.xyz, m.tets, m.phase, D=3e-3, invT2=1e-16, kappa=1e-5)
    fA, fB = np.array([1.0]), np.array([1.0])
    qs = q * np.linspace(0.5, 1.0, nsig)
    gd = np.random.default_rng(2).normal(size=(nsig, 3)) if per_gdir else np.tile((0.2, 1.0, 0.1), (nsig, 1))

    def mat(v):
        return sp.csr_matrix((v, S.col, S.rowptr), shape=(S.ndof, S.ndof))

    real = S.mats["m"] / dt + 0.5 * S.l()
    sc = 1.0 / np.sqrt(mat(real).diagonal())
    u0 = S.initial_condition()
    A, b = [], []
    for j in range(nsig):
        J = qs[j] * S.jg(gd[j])
        A.append(mat(real + 0.5j * J))
        b.append(mat(S.mats["m"] / dt - 0.5 * S.l() - 0.5j * J) @ u0)
    rel = lambda j, u: np.linalg.norm(sc * (b[j] - A[j] @ u)) / np.linalg.norm(sc * b[j])  # noqa: E731
    start = min(rel(j, u0) for j in range(nsig))
    assert start > 1e-9
    ctx = N.Context(0)
    ctx.set_mesh(m.xyz, m.tets, m.phase)
    ctx.set_coeffs(D=3e-3, kappa=1e-5)
    ctx.assemble()
    for part in (0.3, 1e-2, 1e-4):
        rtol = part * start
        _, st = ctx.solve_batched(fA, fB, dt, qs, gd, rtol=rtol, krylov=krylov, guess=1, **opts)
        assert st["iters_total"] >= nsig and (form == 0 or st["precond_used"] == form)
        for j in range(nsig):
            assert rel(j, ctx.solution(j)) <= rtol * (1 + 1e-6) + 1e-14, (part, j)
