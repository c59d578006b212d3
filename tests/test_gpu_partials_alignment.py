"""Block partials are summed by 32-byte loads and refused where their buffer is not aligned for them: solves over
unknown counts of every remainder mod 4, whose scratch buffers follow vectors of that length."""
import numpy as np
import pytest

import dmri_mesh as dm
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("extra", [0, 1, 2, 3])
def test_unknown_counts_of_every_remainder(extra):
    import dmri_native as N

    m = dm.box_mesh((0.0, 0.0, 0.0), (3.0, 2.0, 1.5), 3, 3, 3)
    xyz, tets = m.xyz, m.tets
    for k in range(extra):  # a cell of its own on face 0, 1, 2 of the last cell: one more unknown each
        c = tets[-1].copy()
        face = np.delete(c, k)
        xyz = np.vstack([xyz, xyz[face].mean(0) + 0.3 * (xyz[face].mean(0) - xyz[c[k]])])
        tets = np.vstack([tets, np.r_[face, len(xyz) - 1]]).astype(np.int32)
    ctx = N.Context(0)
    ctx.set_mesh(xyz, tets)
    ctx.set_coeffs(D=3e-3)
    ctx.assemble()
    assert ctx.info()["ndof"] == 64 + extra
    fA, fB = O.gcloud_sequence(O.pgse_piecewise(600.0, 1000.0), 1600.0, 200.0)
    q = O.q_from_b_pgse(2000.0, 10600.0, 43100.0)
    ref, _, _ = O.System(xyz, tets, None, D=3e-3, invT2=1e-16, kappa=0.0).solve((0.0, 1.0, 0.0), q, 200.0, fA, fB,
                                                                               rtol=1e-13)
    for krylov in ("bicgstab", "cocg", "gmres"):
        s, _ = ctx.solve(fA, fB, 200.0, q, (0.0, 1.0, 0.0), rtol=1e-13, krylov=krylov)
        assert abs(s.real - ref) <= 1e-9 * abs(ref)
        sb, _ = ctx.solve_batched(fA, fB, 200.0, [q, 0.5 * q, q], (0.0, 1.0, 0.0), rtol=1e-13, krylov=krylov)
        assert abs(sb[2].real - ref) <= 1e-9 * abs(ref)
