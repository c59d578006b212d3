"""The real part of the operator's entries is held by solves that precondition with it, not by those of the whole
operator: device memory before and after the first solve that takes it, and the same bits whether the entries
came straight from the bounds or through the idle vector."""
import ctypes

import numpy as np
import pytest

import dmri_mesh as dm
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("per_gdir", [False, True])
def test_whole_operator_solves_do_not_hold_the_real_part(per_gdir):
    import dmri_native as N

    nsig = 8
    m = dm.box_mesh((0.0, 0.0, 0.0), (40.0, 40.0, 40.0), 55, 55, 55)
    fA, fB = O.gcloud_sequence(O.pgse_piecewise(600.0, 800.0), 1400.0, 200.0)
    gd = np.random.default_rng(2).normal(size=(nsig, 3)) if per_gdir else (0.2, 1.0, 0.1)

    def free():
        n, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert N.LIB.hipMemGetInfo(ctypes.byref(n), ctypes.byref(total)) == 0
        return n.value

    def context():
        ctx = N.Context(0)
        ctx.set_mesh(m.xyz, m.tets)
        ctx.set_coeffs(D=3e-3)
        ctx.assemble()
        return ctx

    def solve(ctx, q):
        # mapping 6 runs degree 1 of either form: no other buffer comes or goes
        s, st = ctx.solve_batched(fA[:3], fB[:3], 200.0, np.linspace(0.5, 1.0, nsig) * q, gd, rtol=1e-9, mapping=6, lanes=1,
                                  guess=1)
        return s, st["precond_used"], free()

    ctx = context()
    nnz = ctx.info()["nnz"]
    whole, form1, free1 = solve(ctx, 1.2e-4)
    weak, form2, free2 = solve(ctx, 1e-6)
    again, _, free3 = solve(ctx, 1e-6)
    assert (form1, form2) == (1, 2) and nnz > 2_000_000
    assert free1 - free2 >= 0.8 * 8 * nnz and free3 == free2
    assert np.array_equal(weak, again)
    back, _, _ = solve(ctx, 1.2e-4)
    assert np.array_equal(whole, back)
    other, _, _ = solve(context(), 1e-6)
    assert np.array_equal(weak, other)
