"""Uploads and downloads through the pinned buffer, around the sizes where their
route changes: one launch for all parts (up to 2 MB), direct copies, the ring
(from 4 MB; its slots are used again above 8 MB)."""
import threading

import numpy as np
import pytest

from samoa_amd import host, swe

pytestmark = pytest.mark.gpu


def state(n, seed):
    rng = np.random.default_rng(seed)
    s = [rng.normal(0, 1, n) for _ in range(4)]
    s[0][:1], s[3][-1:] = np.nan, np.inf
    return s


def same(got, want):
    return all(x.tobytes() == y.tobytes() for x, y in zip(got, want))


@pytest.mark.parametrize("depth", [0, 1, 8, 14, 15, 16, 17, 18, 19])
def test_round_trip(depth):
    mesh = host.mesh_uniform(depth)
    op = swe.EulerTimestep(mesh)
    for seed in range(3):
        st = state(mesh.n, seed)
        op.upload(*st)
        assert same(op.download(), st)
    # some arrays only, into memory that starts at any byte
    raw = [np.zeros(8 * mesh.n + 16, np.uint8) for _ in range(2)]
    view = [r[3:3 + 8 * mesh.n] for r in raw]
    assert op._lib.swe_download(op._h, None, view[0].ctypes.data, None, view[1].ctypes.data) == 0
    assert same(view, (st[1], st[3]))
    assert not any(r[:3].any() or r[3 + 8 * mesh.n:].any() for r in raw)
    depths, plotter, nbr = op.download_mesh()
    assert np.array_equal(depths, mesh.depth) and np.array_equal(plotter, mesh.plotter)
    assert np.array_equal(nbr.reshape(-1), np.asarray(mesh.nbr).reshape(-1))
    op.close()


@pytest.mark.parametrize("depths", [(0, 3, 1), (9, 4, 12, 9), (17, 2, 16)])
def test_scenarios_of_a_batch(depths):
    meshes = [host.mesh_uniform(d) for d in depths]
    op = swe.Batch(meshes, [dict() for _ in meshes])
    st = [state(m.n, i) for i, m in enumerate(meshes)]
    for i, s in enumerate(st):
        op.upload(i, *s)
    for i, s in reversed(list(enumerate(st))):
        assert same(op.download(i), s)
    op.close()


@pytest.mark.parametrize("depth", [0, 8, 13, 20, 21])
def test_traversal_returns_the_flags(depth):
    """The flags and results of swe_step against those left on the device."""
    mesh = host.mesh_uniform(depth)
    eta, _, _, b = host.tsunami(mesh, seed=5, drytol=1e-3)
    z = np.zeros(mesh.n)
    got = []
    for flags in (True, False):
        op = swe.EulerTimestep(mesh, scaling=1.0e6, dry_tolerance=1e-3, min_depth=max(depth - 1, 0),
                               max_depth=depth + 1)
        op.upload(eta, z, z, b)
        dt = 1e-9
        for fwd in (True, False):
            r = op.traverse(dt, fwd, flags=flags)
            dt = 0.45 * r.dt_cfl
        got.append((r.dt_cfl, r.n_refine, op.download()))
        if flags:
            assert np.isin(r.refine, (-1, 0, 1)).all() and (r.refine == 1).sum() == r.n_refine
        op.close()
    assert got[0][:2] == got[1][:2] and same(got[0][2], got[1][2])


def test_two_threads_download_at_once():
    mesh = host.mesh_uniform(17)
    ops, errors = [swe.EulerTimestep(mesh) for _ in range(2)], []

    def work(i):
        for k in range(4):
            st = state(mesh.n, 10 * i + k)
            ops[i].upload(*st)
            if not same(ops[i].download(), st):
                errors.append((i, k))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for op in ops:
        op.close()
    assert not errors
