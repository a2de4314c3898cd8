"""Steps with stored edge lists against steps whose workgroups build them: a
remeshed handle builds its own for the first two traversals and stores them
for the following ones; a new handle on the same mesh has them from the start."""
import numpy as np
import pytest

from samoa_amd import host, swe

pytestmark = pytest.mark.gpu


def pair(depth, chunk, **params):
    rng = np.random.default_rng(depth + chunk)
    mesh = host.mesh_uniform(depth)
    kw = dict(scaling=1000.0, dry_tolerance=1e-3, min_depth=max(depth - 1, 0), max_depth=depth + 2,
              **params)
    old = swe.EulerTimestep(mesh, **kw)
    old.set_tuning(chunk, 0)
    b = -5.0 + 6.0 * rng.random(mesh.n)
    eta = np.maximum(0.2 * rng.normal(0, 1, mesh.n), b)
    h = eta - b
    old.upload(eta, h * rng.normal(0, 0.5, mesh.n), h * rng.normal(0, 0.5, mesh.n), b)
    old.adapt((rng.random(mesh.n) < 0.3).astype(np.int8))
    new = swe.EulerTimestep(swe.Mesh(*old.download_mesh()), **kw)
    new.set_tuning(chunk, 0)
    new.upload(*old.download())
    return old, new


@pytest.mark.parametrize("chunk", [128, 256, 512])
@pytest.mark.parametrize("depth", [0, 5, 9, 12])
@pytest.mark.parametrize("form", ["augmented", "fwave", "toleranced", "jumps", "llf", "walls"])
def test_same_steps(depth, chunk, form):
    params = {"fwave": dict(solver=swe.SOLVER_FWAVE), "llf": dict(solver=swe.SOLVER_LLF_BATH),
              "walls": dict(boundary=swe.BC_WALL)}.get(form, {})
    ops = pair(depth, chunk, **params)
    dt = [1e-3, 1e-3]
    for op in ops:
        if form == "toleranced":
            op.set_arithmetic(swe.ARITH_TOLERANCED)
        if form == "jumps":
            op.keep_eta_jump_flags(0.1, 0.01)
    for fwd in (True, False, False, True, True, False):
        r = [op.traverse(x, fwd, flags=True) for op, x in zip(ops, dt)]
        assert r[0].dt_cfl == r[1].dt_cfl and r[0].n_refine == r[1].n_refine
        assert np.array_equal(r[0].refine, r[1].refine)
        dt = [0.45 * x.dt_cfl for x in r]
        for x, y in zip(*(op.download() for op in ops)):
            assert np.array_equal(x, y)
    for steps in (1, 2, 9):
        t = [op.run(steps, x, True) for op, x in zip(ops, dt)]
        assert t[0] == t[1]
        for x, y in zip(*(op.download() for op in ops)):
            assert np.array_equal(x, y)
    for op in ops:
        op.close()


def test_a_run_after_remeshing_stores_the_lists():
    """The first run on a changed mesh, in one call and in two."""
    for first in (9, 2):
        old, new = pair(9, 256)
        got = [op.run(first, 1e-3, True) for op in (old, new)]
        if first == 2:
            got = [op.run(7, dt, True, time=t) for op, (t, dt) in zip((old, new), got)]
        assert got[0] == got[1]
        for x, y in zip(old.download(), new.download()):
            assert np.array_equal(x, y)
        old.close()
        new.close()
