"""Set-up rows at the edges of their register sorts: incidence lists of 32 cells and more, rows of up to 256
candidate columns and beyond (left to the LDS kernel), with and without an interface through them."""
import numpy as np
import pytest

import dmri_mesh as dm
import oracle as O

pytestmark = pytest.mark.gpu


def _fan(n, two):
    """n cells around the edge from vertex 0 to vertex 1; two: the phase changes half way around."""
    a = 2 * np.pi * np.arange(n) / n
    ring = np.stack([np.cos(a), np.sin(a), 0.1 * np.sin(3 * a)], 1)
    xyz = np.concatenate([[[0, 0, -0.5], [0, 0, 1.0]], ring])
    tets = np.array([[0, 1, 2 + i, 2 + (i + 1) % n] for i in range(n)], np.int32)
    return xyz, tets, (np.arange(n) < n // 2).astype(np.int32) if two else None


@pytest.mark.parametrize("two", [False, True])
@pytest.mark.parametrize("n", [3, 8, 31, 32, 33, 62, 64, 65, 130, 400, "cylinder", "box"])
def test_pattern_and_matrices_match_oracle(n, two):
    import dmri_native as N

    if n == "cylinder":
        m = dm.cylinder_mesh(5.0, 5.0, 5000, seed=1, interface_radii=(2.5,) if two else ())
        xyz, tets, phase = m.xyz, m.tets, m.phase
    elif n == "box":
        m = dm.box_mesh((0, 0, 0), (1, 1, 1), 9, 7, 5)
        xyz, tets = m.xyz, m.tets
        # a chequered phase: interface facets at every vertex
        phase = (np.floor(9 * xyz[tets].mean(1)).sum(1) % 2).astype(np.int32) if two else None
    else:
        xyz, tets, phase = _fan(n, two)
    ctx = N.Context(0)
    ctx.set_mesh(xyz, tets, phase)
    ctx.set_coeffs(D=3e-3, kappa=2e-5)
    ctx.assemble()
    S = O.System(xyz, tets, phase, D=3e-3, invT2=1e-16, kappa=2e-5)
    rowptr, col, dof_of = ctx.export_pattern()
    assert np.array_equal(rowptr, S.rowptr) and np.array_equal(col, S.col)
    for name in ("m", "k", "gi", "jx"):
        ref = S.mats[name]
        assert np.max(np.abs(ctx.export_values(name) - ref)) <= 1e-13 * max(np.max(np.abs(ref)), 1e-300), name
    fA, fB = O.gcloud_sequence(O.pgse_piecewise(400.0, 600.0), 1000.0, 200.0)
    s, _ = ctx.solve(fA, fB, 200.0, 1e-4, (0.3, 1.0, 0.2), rtol=1e-13)
    ref, _, _ = S.solve((0.3, 1.0, 0.2), 1e-4, 200.0, fA, fB, rtol=1e-13)
    assert abs(s.real - ref) <= 1e-9 * abs(ref)
