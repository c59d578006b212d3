"""The SpMV mapping follows the form of the preconditioner: a tuned choice (dmri_set_tuning, a line of a tuning
database) that cannot run the form a solve takes gives way to the default mapping, a mapping the caller
names stays, and the default of a wide launch group of one direction changes with its rows."""
import numpy as np
import pytest

import dmri_mesh as dm
import oracle as O

pytestmark = pytest.mark.gpu


def _context(nv, kind="cylinder"):
    import dmri_native as N

    m = (dm.neuron_mesh(target_nv=nv, seed=3) if kind == "neuron"
         else dm.cylinder_mesh(6.0, 6.0, nv, seed=8, interface_radii=(3.0,)))
    ctx = N.Context(0)
    ctx.set_mesh(m.xyz, m.tets, m.phase)
    ctx.set_coeffs(D=3e-3, kappa=1e-5 if m.phase is not None else 0.0)
    ctx.assemble()
    return ctx


def _args(nsig, q=2e-5):
    fA, fB = O.gcloud_sequence(O.pgse_piecewise(600.0, 800.0), 1400.0, 200.0)
    return fA, fB, 200.0, np.linspace(0.3, 1.0, nsig) * q, (0.2, 1.0, 0.1)


@pytest.mark.parametrize("kind,nv,nsig,krylov,q,form", [
    ("cylinder", 6000, 12, "bicgstab", 2e-5, 2), ("cylinder", 1000, 5, "gmres", 2e-5, 2),
    ("cylinder", 1000, 18, "gmres", 2e-5, 2), ("neuron", 4000, 20, "bicgstab", 2e-2, 3)])
def test_tuned_mapping_keeps_the_form(kind, nv, nsig, krylov, q, form, tmp_path):
    ctx = _context(nv, kind)
    args = _args(nsig, q)
    kw = dict(rtol=1e-12, krylov=krylov)
    a, st = ctx.solve_batched(*args, **kw)
    assert st["precond_used"] == form
    for mapping in (4, 6) if form == 2 else (4,):
        ctx.set_tuning(nsig, False, 1, mapping)
        b, sb = ctx.solve_batched(*args, **kw)
        assert sb["precond_used"] == form and sb["iters_total"] == st["iters_total"]
        assert np.array_equal(a, b)
    if form == 2:  # a mapping the caller names is taken as it is (without the complex diagonal it may not converge)
        c, sc = ctx.solve_batched(*args, mapping=4, lanes=1, **kw)
        assert sc["iters_total"] > 1.3 * st["iters_total"]
        assert np.max(np.abs(a - c)) <= 1e-9
    # the same choice from a line of a tuning database
    db = tmp_path / "tune.db"
    ctx.tune_db(db, nsig, False)
    line = db.read_text().split()
    line[5:7] = ["4", "1"]
    db.write_text(" ".join(line) + "\n")
    assert ctx.tune_db(db, nsig, False) == ((4, 1), True)
    b, sb = ctx.solve_batched(*args, **kw)
    assert sb["iters_total"] == st["iters_total"] and np.array_equal(a, b)


@pytest.mark.parametrize("nv,nsig,precond,krylov,mapping", [
    (1000, 16, 0, 0, 2), (1000, 17, 0, 0, 4), (1000, 32, 0, 0, 4), (1000, 32, 1, 0, 4), (1000, 64, 0, 0, 4),
    (11000, 17, 0, 0, 2), (30000, 48, 0, 0, 2), (6000, 40, 1, 0, 4), (1000, 40, 0, 1, 2), (1000, 41, 0, 1, 4),
    (5000, 48, 0, 1, 2)])
def test_default_of_wide_groups(nv, nsig, precond, krylov, mapping):
    ctx = _context(nv)
    args = _args(nsig)
    kw = dict(rtol=1e-12, precond=precond, krylov=krylov)
    a, sa = ctx.solve_batched(*args, **kw)
    b, sb = ctx.solve_batched(*args, mapping=mapping, lanes=1, **kw)
    c, _ = ctx.solve_batched(*args, mapping=6 - mapping, lanes=1, **kw)
    assert sa["iters_total"] == sb["iters_total"] and np.array_equal(a, b) and not np.array_equal(a, c)
    assert np.max(np.abs(a - c)) <= 1e-9
