"""A mesh whose few cells use the last of very many vertices: 32 lanes per incidence list are more threads than one
launch holds, the other vertices take part in nothing."""
import numpy as np
import pytest

import dmri_mesh as dm
import oracle as O

pytestmark = pytest.mark.gpu


def test_more_lists_than_a_launch_has_groups():
    import dmri_native as N

    m = dm.box_mesh((0.0, 0.0, 0.0), (3.0, 2.0, 1.5), 3, 3, 3)
    nv = 2**32 // 32 + 5000
    xyz = np.zeros((nv, 3))
    at = np.r_[0:10, nv - m.nv + 10 : nv]  # the first ten vertices first, the rest last
    xyz[at] = m.xyz
    fA, fB = O.gcloud_sequence(O.pgse_piecewise(600.0, 1000.0), 1600.0, 200.0)
    q = O.q_from_b_pgse(2000.0, 10600.0, 43100.0)
    out = []
    for x, t in ((m.xyz, m.tets), (xyz, at.astype(np.int32)[m.tets])):
        ctx = N.Context(0)
        ctx.set_mesh(x, t)
        ctx.set_coeffs(D=3e-3)
        ctx.assemble()
        s, _ = ctx.solve(fA, fB, 200.0, q, (0.0, 1.0, 0.0), rtol=1e-13)
        out.append((ctx.info()["ndof"], ctx.info()["nnz"], s, ctx.solution()))
        ctx.close()
    assert out[0][:3] == out[1][:3] and np.array_equal(out[0][3], out[1][3])
