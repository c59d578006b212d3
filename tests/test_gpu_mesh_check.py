"""The device checks of dmri_mesh_set: what they refuse, in which order, the sizes they report, and that
a refused mesh leaves the context's mesh as it was."""
import numpy as np
import pytest

import dmri_mesh as dm

pytestmark = pytest.mark.gpu


def _set(ctx, xyz, tets, phase=None):
    import dmri_native as N

    with pytest.raises(N.DmriError) as e:
        ctx.set_mesh(xyz, tets, phase)
    assert e.value.code == -5
    return str(e.value)


@pytest.mark.parametrize("n", [1, 5, 12])
def test_refusals_and_sizes(n):
    import dmri_native as N

    m = dm.box_mesh((0.0, 0.0, 0.0), (3.0, 2.0, 1.5), n, n, n)
    phase = (np.arange(m.nc) % 2).astype(np.int32)
    ctx = N.Context(0)
    ctx.set_mesh(m.xyz, m.tets, phase)
    last = m.nc - 1
    for cell in (0, last):
        for bad in (-1, m.nv, 2**30):
            t = m.tets.copy()
            t[cell, 3] = bad
            x = m.xyz.copy()
            x[0, 1] = np.nan  # the vertex range is reported first
            assert f"cell {cell} has a vertex index out of range" in _set(ctx, x, t)
        t = m.tets.copy()
        t[cell] = t[cell, 0]
        assert f"degenerate cell {cell}" in _set(ctx, m.xyz, t)
        p = phase.copy()
        p[cell] = 2
        assert "cell phase must be 0 or 1" in _set(ctx, m.xyz, t, p)
    for v, value in ((0, np.inf), (m.nv - 1, np.nan)):
        x = m.xyz.copy()
        x[v, 2] = value
        assert "non-finite coordinate" in _set(ctx, x, m.tets)
    ctx.set_coeffs(D=3e-3)
    ctx.assemble()
    info = ctx.info()
    hmin, hmax = m.hminmax()
    assert (info["nv"], info["nc"], info["ncomp"]) == (m.nv, m.nc, 2)
    assert info["hmin"] == pytest.approx(hmin, rel=4e-16) and info["hmax"] == pytest.approx(hmax, rel=4e-16)
