"""SpMV rows straight from global memory (mapping 1) on 4 to 32 lanes: several tiles per block and a single
one, rows longer than a lane's entries in flight, a last tile cut short; against the staged rows."""
import numpy as np
import pytest

import dmri_mesh as dm
import oracle as O

pytestmark = pytest.mark.gpu


def _fan(n):
    """A vertex on the axis shared by every cell of a fan: one row as long as the mesh."""
    a = 2 * np.pi * np.arange(n) / n
    ring = np.stack([np.cos(a), np.sin(a), 0.1 * np.sin(3 * a)], 1)
    xyz = np.concatenate([[[0, 0, 0.0], [0, 0, 1.0]], ring])
    tets = np.array([[0, 1, 2 + i, 2 + (i + 1) % n] for i in range(n)], np.int32)
    return dm.TetMesh(xyz, tets)


@pytest.mark.parametrize("lanes", [4, 8, 16, 32])
@pytest.mark.parametrize("krylov", ["bicgstab", "cocg"])
@pytest.mark.parametrize("mesh", ["fan", "small", "large"])
def test_direct_rows_match_staged(mesh, krylov, lanes):
    import dmri_native as N

    m = _fan(60) if mesh == "fan" else dm.cylinder_mesh(6.0, 6.0, 1500 if mesh == "small" else 70001, seed=5)
    fA, fB = O.gcloud_sequence(O.pgse_piecewise(600.0, 1000.0), 1600.0, 400.0)
    q = np.array([O.q_from_b_pgse(3000.0, 10600.0, 43100.0)])
    ctx = N.Context(0)
    ctx.set_mesh(m.xyz, m.tets)
    ctx.set_coeffs(D=3e-3)
    ctx.assemble()
    a, _ = ctx.solve_batched(fA, fB, 400.0, q, (0.3, 1.0, 0.2), rtol=1e-13, krylov=krylov, mapping=1, lanes=lanes)
    ua = ctx.solution()
    b, _ = ctx.solve_batched(fA, fB, 400.0, q, (0.3, 1.0, 0.2), rtol=1e-13, krylov=krylov, mapping=2, lanes=4)
    assert abs(a[0] - b[0]) <= 1e-11 * abs(b[0])
    assert np.linalg.norm(ua - ctx.solution()) <= 1e-10 * np.linalg.norm(ua)
