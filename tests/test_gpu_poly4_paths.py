"""The degree-4 polynomial of the real part on the ways around a plain solve: captured runs, timed iterations, an
iteration limit that is met while a run's last iteration stands at its test, the resumable batch, and the
strong periodic form."""
import numpy as np
import pytest

import dmri_mesh as dm
import dmri_sequences as DS
import oracle as O

pytestmark = pytest.mark.gpu

CASES = [("cocg", 1, 45000), ("cocg", 3, 3000), ("cocg", -4, 3000), ("bicgstab", 1, 45000), ("bicgstab", 5, 9000),
         ("bicgstab", -5, 9000)]


def _problem(nsig, nv, dt=400.0):
    import dmri_native as N

    per_gdir, nsig = nsig < 0, abs(nsig)
    m = dm.cylinder_mesh(6.0, 6.0, nv, seed=8, interface_radii=(3.0,))
    fA, fB = O.gcloud_sequence(O.pgse_piecewise(3 * dt, 4 * dt), 7 * dt, dt)
    qs = np.linspace(0.3, 1.0, nsig) * 2e-5 * 400.0 / dt
    gd = np.random.default_rng(2).normal(size=(nsig, 3)) if per_gdir else (0.2, 1.0, 0.1)
    ctx = N.Context(0)
    ctx.set_mesh(m.xyz, m.tets, m.phase)
    ctx.set_coeffs(D=3e-3, kappa=1e-5)
    ctx.assemble()
    return ctx, (fA, fB, dt, qs, gd)


@pytest.mark.parametrize("krylov,nsig,nv", CASES)
def test_graphs_timed_iterations_and_batches(krylov, nsig, nv):
    ctx, args = _problem(nsig, nv)
    kw = dict(rtol=1e-12, krylov=krylov)
    a, st = ctx.solve_batched(*args, snap_every=1, **kw)
    assert st["precond_used"] == 2
    for more in (dict(graphs=1), dict(profile=3), dict(graphs=1, profile=2)):
        b, sb = ctx.solve_batched(*args, snap_every=1, **more, **kw)
        assert np.array_equal(a, b) and np.array_equal(st["snapshots"], sb["snapshots"]), more
        assert sb["iters_total"] == st["iters_total"]
        assert (sb["graph_launches"] > 0) == ("graphs" in more)
        if "profile" in more:  # four steps of the polynomial stand in one entry
            assert sb["kern_launches"][1] > 0 and sb["kern_ms"][1] > 0
    for graphs in (0, 1):
        with ctx.batch(*args, graphs=graphs, **kw) as b:
            for piece in (1, 2, len(args[0]) - 3):
                b.advance(piece)
                ctx.solve_batched(*args, **kw)  # other work of the context in between
            sig, steps = b.signals()
        assert steps == len(args[0]) and np.array_equal(sig, a)


@pytest.mark.parametrize("krylov,nsig,nv", CASES)
def test_iteration_limit(krylov, nsig, nv):
    import dmri_native as N

    ctx, args = _problem(nsig, nv, dt=2000.0)
    kw = dict(rtol=1e-12, krylov=krylov)
    a, st = ctx.solve_batched(*args, **kw)
    assert st["precond_used"] == 2 and st["iters_max"] > 9
    # below, at and above the first run's length (8), and one short of what the worst step takes
    for maxit in (1, 7, 8, 9, st["iters_max"] - 1):
        for graphs in (0, 1):
            with pytest.raises(N.DmriError) as e:
                ctx.solve_batched(*args, maxit=maxit, graphs=graphs, **kw)
            assert e.value.code == -4
    b, _ = ctx.solve_batched(*args, maxit=st["iters_max"], **kw)
    assert np.array_equal(a, b)


@pytest.mark.parametrize("nsig", [1, 2])
def test_strong_periodic(nsig):
    import dmri_native as N

    dt, T = 400.0, 2400.0
    fA, fB, FB = DS.gcloud_loop(DS.pgse(400.0, 2000.0), T, dt, DS.pgse_integral(400.0, 2000.0))
    FA = DS.gcloud_loop(DS.pgse_integral(400.0, 2000.0), T, dt)[0]
    n = 36 if nsig == 1 else 29  # more than 40000 values
    m = dm.box_mesh((0.0, 0.0, 0.0), (4.0, 3.0, 3.0), n, n, n)
    ctx = N.Context(0)
    ctx.set_mesh(m.xyz, m.tets)
    ctx.set_coeffs(D=2e-3)
    ctx.set_periodic_strong((1, 1, 0))
    ctx.assemble()
    assert ctx.info()["ndof"] * nsig > 40000
    kw = dict(rtol=1e-13, F_explicit=FB, F_implicit=FA)
    q = 1e-5
    gd = [(1.0, 0.4, 0.2), (0.1, 1.0, 0.5)][:nsig]
    a, st = ctx.solve_batched(fA, fB, dt, [q] * nsig, gd, **kw)
    b, sj = ctx.solve_batched(fA, fB, dt, [q] * nsig, gd, precond=1, **kw)
    assert st["precond_used"] == 2 and 2 * st["iters_total"] < sj["iters_total"]
    assert np.max(np.abs(a - b)) <= 1e-11
    g1, sg = ctx.solve_batched(fA, fB, dt, [q] * nsig, gd, graphs=1, **kw)
    assert sg["graph_launches"] > 0 and np.array_equal(a, g1)
