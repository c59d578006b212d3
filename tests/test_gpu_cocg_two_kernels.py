"""COCG's two-kernel iteration (one signal: update of r and p-step both folded in): repeated solves bit for
bit alike, graph replay as plain launches, the oracle's signal, and the iterate of a solve stopped by a
loose tolerance within that tolerance (its last x += alpha p is applied by the kernel that stops it)."""
import numpy as np
import pytest

import dmri_mesh as dm
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nv,steps", [(130, 5), (2500, 8), (20000, 6)])
def test_two_kernel_iterations(nv, steps):
    import dmri_native as N

    m = dm.cylinder_mesh(6.0, 6.0, nv, seed=4, interface_radii=(3.0,))
    fA, fB = O.gcloud_sequence(O.pgse_piecewise(600.0, 1000.0), 1600.0, 200.0)
    fA, fB = fA[:steps], fB[:steps]
    q = O.q_from_b_pgse(3000.0, 10600.0, 43100.0)
    g = (0.2, 1.0, 0.1)
    ctx = N.Context(0)
    ctx.set_mesh(m.xyz, m.tets, m.phase)
    ctx.set_coeffs(D=3e-3, kappa=1e-5)
    ctx.assemble()
    a, st = ctx.solve(fA, fB, 200.0, q, g, rtol=1e-13, krylov="cocg")
    ua = ctx.solution()
    b, _ = ctx.solve(fA, fB, 200.0, q, g, rtol=1e-13, krylov="cocg")
    ub = ctx.solution()
    c, _ = ctx.solve(fA, fB, 200.0, q, g, rtol=1e-13, krylov="cocg", graphs=1)
    assert a == b == c and np.array_equal(ua, ub) and st["restarts"] == 0
    S = O.System(m.xyz, m.tets, m.phase, D=3e-3, invT2=1e-16, kappa=1e-5)
    ref, _, _ = S.solve(g, q, 200.0, fA, fB, rtol=1e-13)
    assert abs(a.real - ref) <= 1e-9 * abs(ref)
    ctx.solve(fA[:1], fB[:1], 200.0, q, g, rtol=1e-3, krylov="cocg", guess=1)
    loose = ctx.solution()
    ctx.solve(fA[:1], fB[:1], 200.0, q, g, rtol=1e-13, krylov="cocg", guess=1)
    tight = ctx.solution()
    # the condition number of the step's operator is below 1e2 on these meshes
    assert 0 < np.linalg.norm(loose - tight) <= 1e-1 * np.linalg.norm(tight)
