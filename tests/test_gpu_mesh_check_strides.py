"""The device checks of dmri_mesh_set over meshes with more cells and vertices than one pass of the grid covers
(1024 blocks of 256 threads), and the sizes of cells whose squared size is out of the usual range."""
import numpy as np
import pytest

import dmri_mesh as dm

pytestmark = pytest.mark.gpu
STRIDE = 1024 * 256


def _refused(ctx, xyz, tets, phase=None):
    import dmri_native as N

    with pytest.raises(N.DmriError) as e:
        ctx.set_mesh(xyz, tets, phase)
    assert e.value.code == -5
    return str(e.value)


def test_checks_carry_over_strides():
    import dmri_native as N

    m = dm.box_mesh((0.0, 0.0, 0.0), (3.0, 2.0, 1.5), 65, 65, 65)
    assert m.nv > STRIDE and m.nc > 6 * STRIDE
    ctx = N.Context(0)
    xyz = m.xyz.copy()
    xyz[-1] += (0.5, 0.25, 0.125)  # the last vertex of all stretches the last cells
    ctx.set_mesh(xyz, m.tets)
    E = np.max([np.linalg.norm(xyz[m.tets[:, a]] - xyz[m.tets[:, b]], axis=1) for a in range(4) for b in range(a)],
               axis=0)
    info = ctx.info()
    assert info["hmin"] == pytest.approx(E.min(), rel=4e-16) and info["hmax"] == pytest.approx(E.max(), rel=4e-16)
    assert E.argmax() >= STRIDE
    for first, other in ((m.nc - 1, None), (STRIDE + 7, 3 * STRIDE + 7), (STRIDE - 1, STRIDE), (7, 5 * STRIDE + 7)):
        bad = [c for c in (first, other) if c is not None]
        t = m.tets.copy()
        t[bad, 2] = m.nv
        assert f"cell {first} has a vertex index out of range" in _refused(ctx, m.xyz, t)
        t = m.tets.copy()
        t[bad] = t[bad, :1]
        assert f"degenerate cell {first}" in _refused(ctx, m.xyz, t)
        p = np.zeros(m.nc, np.int32)
        p[bad] = -1
        assert "cell phase must be 0 or 1" in _refused(ctx, m.xyz, m.tets, p)
    for v in (m.nv - 1, STRIDE + 3):
        x = m.xyz.copy()
        x[v, 1] = np.inf
        assert "non-finite coordinate" in _refused(ctx, x, m.tets)
    info = ctx.info()  # the refusals left the first mesh
    assert info["hmax"] == pytest.approx(E.max(), rel=4e-16)


@pytest.mark.parametrize("scale", [1e-150, 1e149, 1e152, 1e153])
def test_sizes_of_extreme_cells(scale):
    import dmri_native as N

    m = dm.box_mesh((0.0, 0.0, 0.0), (3.0, 2.0, 1.5), 2, 3, 2)
    hmin, hmax = m.hminmax()
    ctx = N.Context(0)
    ctx.set_mesh(scale * m.xyz, m.tets)
    info = ctx.info()
    assert info["hmin"] == pytest.approx(scale * hmin, rel=1e-14)
    assert info["hmax"] == pytest.approx(scale * hmax, rel=1e-14)
