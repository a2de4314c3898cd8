"""The device dt chain of swe_run / swe_batch_run, whose steps form their dt
from the previous step's partials on small meshes and from the finalize
kernel on large ones, against the host's chain of single traversals: states,
time and dt bit for bit, however the steps are split over calls."""
import numpy as np
import pytest

from samoa_amd import host, swe

pytestmark = pytest.mark.gpu

COURANT = 0.45


def beach(mesh, seed=0):
    rng = np.random.default_rng(seed)
    cen = mesh.centroids()
    b = -8.0 + 11.0 * cen[:, 0] + 0.5 * np.sin(9.0 * cen[:, 1])
    eta = np.where(np.hypot(cen[:, 0] - 0.3, cen[:, 1] - 0.5) < 0.2, 1.0 + rng.random(), 0.0)
    eta = np.where(eta > b + 1e-3, eta, np.minimum(b, 0.0))
    z = np.zeros(mesh.n)
    return eta, z, z.copy(), b


def operator(mesh, chunk=None):
    op = swe.EulerTimestep(mesh, scaling=1e3, dry_tolerance=1e-3, courant=COURANT,
                           boundary=swe.BC_WALL)
    if chunk:
        op.set_tuning(chunk, 0)
    return op


class HostChain:
    """dt and time as pre/post_traversal_grid_op keep them on the host."""

    def __init__(self, mesh, st, dt0):
        self.op = operator(mesh)
        self.op.upload(*st)
        self.dt, self.t, self.fwd = dt0, 0.0, False

    def run(self, n, clamp=-1.0):
        for _ in range(n):
            res = self.op.traverse(self.dt, self.fwd)
            self.t = self.t + self.dt
            self.dt = COURANT * res.dt_cfl
            if clamp > 0.0:
                self.dt = min(clamp, self.dt)
            self.fwd = not self.fwd


# one chunk, ragged, few chunks; the largest chain (1024 chunks of 256 cells);
# the smallest (2048) and largest (4096) meshes whose workgroups meet, and,
# with 128-cell chunks, one with a finalize kernel (8192)
@pytest.mark.parametrize("depth,chunk", [(0, None), (5, None), (7, 128), (10, 512), (12, None),
                                         (17, None), (18, None), (18, 128), (19, 128)])
@pytest.mark.parametrize("parts", [[5], [1, 4], [2, 3], [1, 1, 1, 1, 1]])
def test_pieces_of_a_run_equal_single_traversals(depth, chunk, parts):
    print("case:", depth, chunk, parts, flush=True)
    mesh = host.mesh_uniform(depth)
    st = beach(mesh)
    dt0 = host.initial_dt(mesh, st, COURANT) * 1e3
    ref = HostChain(mesh, st, dt0)
    op = operator(mesh, chunk)
    op.upload(*st)
    fwd = False
    for i, n in enumerate(parts):
        wait = i % 2 == 0
        got = op.run(n, dt0 if i == 0 else None, fwd, wait=wait)
        ref.run(n)
        fwd ^= n % 2 == 1
        if wait:
            assert got == (ref.t, ref.dt)
    assert op.run(0, None, fwd) == (ref.t, ref.dt)
    for a, b in zip(op.download(), ref.op.download()):
        assert np.array_equal(a, b)
    op.close()
    ref.op.close()


def test_other_calls_between_the_pieces():
    """A clamp that changes, single traversals, a launch shape, a stream and
    a device-pointer traversal between the pieces leave the chain alone."""
    import torch

    mesh = host.mesh_uniform(11)
    st = beach(mesh, 1)
    dt0 = host.initial_dt(mesh, st, COURANT) * 1e3
    ref = HostChain(mesh, st, dt0)
    op = operator(mesh)
    op.upload(*st)
    op.run(7, dt0, False)
    ref.run(7)
    # the dt the run left holds, whatever the next run's clamp is
    clamp = 0.5 * ref.dt
    op.run(4, None, True, dt_clamp=clamp, wait=False)
    ref.run(4, clamp)
    op.set_tuning(128, 0)
    op.run(3, None, True, dt_clamp=clamp, wait=False)
    ref.run(3, clamp)
    stream = torch.cuda.Stream()
    op.set_stream(stream.cuda_stream)
    q = [torch.tensor(a, device="cuda") for a in st]
    o = [torch.empty_like(q[0]) for _ in range(3)]
    cfl = torch.zeros(1, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    op.step_device(*[a.data_ptr() for a in q + o], 1e-3, True, cfl.data_ptr(),
                   stream=stream.cuda_stream)
    op.run(2, None, False, dt_clamp=clamp, wait=False)
    ref.run(2, clamp)
    # a traversal with the host's dt moves the state, not the device's chain
    one = op.traverse(0.25 * ref.dt, False)
    assert one.dt_cfl == ref.op.traverse(0.25 * ref.dt, False).dt_cfl
    ref.fwd = True
    op.run(3, None, True, dt_clamp=clamp, wait=False)
    ref.run(3, clamp)
    assert op.run(0, None, False, dt_clamp=clamp) == (ref.t, ref.dt)
    for a, b in zip(op.download(), ref.op.download()):
        assert np.array_equal(a, b)
    op.close()
    ref.op.close()


def test_remeshing_between_the_pieces():
    """The step after a remeshing forms its dt from the old mesh's partials,
    also where the new mesh needs more room or leaves the chain's range."""
    for depth, dmax in ((6, 9), (16, 18), (18, 20)):
        print("case:", depth, flush=True)
        mesh = host.mesh_uniform(depth)
        st = beach(mesh, 2)
        dt = host.initial_dt(mesh, st, COURANT) * 1e3
        ops = [swe.EulerTimestep(mesh, scaling=1e3, dry_tolerance=1e-3, courant=COURANT,
                                 min_depth=depth - 1, max_depth=dmax, boundary=swe.BC_WALL)
               for _ in range(2)]
        for op in ops:
            op.upload(*st)
        rng = np.random.default_rng(depth)
        t, fwd = 0.0, False
        for k in range(4):
            ops[0].run(3, dt if k == 0 else None, fwd, wait=k == 0)
            for _ in range(3):
                res = ops[1].traverse(dt, fwd)
                t, dt, fwd = t + dt, COURANT * res.dt_cfl, not fwd
            flags = (rng.random(ops[0].n) < 0.6).astype(np.int8) - (rng.random(ops[0].n) < 0.1)
            n = [op.adapt(flags.astype(np.int8))[0] for op in ops]
            assert n[0] == n[1]
            fwd = not fwd
        assert ops[0].run(0, None, fwd) == (t, dt)
        for a, b in zip(ops[0].download(), ops[1].download()):
            assert np.array_equal(a, b)
        for op in ops:
            op.close()


def test_batch_of_uneven_meshes():
    depths = [0, 9, 5, 12, 11]
    meshes = [host.mesh_uniform(d) for d in depths]
    states = [beach(m, i) for i, m in enumerate(meshes)]
    dt0 = [host.initial_dt(m, s, COURANT) * 1e3 for m, s in zip(meshes, states)]
    b = swe.Batch(meshes, [dict(scaling=1e3, dry_tolerance=1e-3, courant=COURANT,
                                boundary=swe.BC_WALL) for _ in meshes])
    refs = []
    for i, (m, s) in enumerate(zip(meshes, states)):
        b.upload(i, *s)
        refs.append(HostChain(m, s, dt0[i]))
    t, dt = b.run(5, dt0, False)
    t, dt = b.run(4, dt, True, time=t)
    for i, r in enumerate(refs):
        r.run(9)
        assert (t[i], dt[i]) == (r.t, r.dt)
        for x, y in zip(b.download(i), r.op.download()):
            assert np.array_equal(x, y)
        r.op.close()
    b.close()


# cells per chunk x chunks around the number of places workgroups meet at
@pytest.mark.parametrize("grid", [0, 8])
@pytest.mark.parametrize("depth,chunk", [(3, 128), (11, 256), (11, 128), (12, 512), (14, 256),
                                         (19, 256), (19, 128)])
def test_single_steps_publish_their_results(depth, chunk, grid):
    """dt_cfl and the refinement count of repeated steps do not depend on how
    the workgroups' partials are reduced: equal to the counted flags and to
    the other launch shapes', with the places left clean for the next step."""
    print("case:", depth, chunk, grid, flush=True)
    meshes = [host.mesh_uniform(depth)]
    op = swe.EulerTimestep(meshes[0], scaling=1e3, dry_tolerance=1e-3, min_depth=depth - 1,
                           max_depth=depth + 6, boundary=swe.BC_WALL)
    st = beach(meshes[0], 5)
    dt = 0.4 * host.initial_dt(meshes[0], st, COURANT) * 1e3
    got = []
    for c, g in ((chunk, grid), (256, 0), (512, 16)):
        op.set_tuning(c, g)
        op.upload(*st)
        rows = []
        for k in range(3):
            res = op.traverse(dt, k % 2 == 0, flags=True)
            assert res.n_refine == int((res.refine == 1).sum())
            rows.append((res.dt_cfl, res.n_refine))
        got.append(rows)
    assert got[0] == got[1] == got[2]
    assert depth < 8 or got[0][0][1] > 0
    op.close()


def test_cells_without_numbers_set_no_limit():
    """NaN cells are left out of the CFL minimum, as a comparison with NaN
    leaves them out in the reference's reduction; without any other cell it
    is huge."""
    mesh = host.mesh_uniform(9)
    st = beach(mesh, 3)
    op = operator(mesh)
    op.upload(*st)
    whole = op.traverse(1e-3, True).dt_cfl
    bad = [a.copy() for a in st]
    bad[1][::97] = np.nan
    op.upload(*bad)
    assert whole <= op.traverse(1e-3, True).dt_cfl < np.inf
    huge = np.finfo(float).max
    for k in range(4):
        bad = [a.copy() for a in st]
        bad[k][:] = np.nan
        op.upload(*bad)
        assert op.traverse(1e-3, True).dt_cfl == huge
        op.upload(*bad)
        assert op.run(3, 1e-3, True)[1] == COURANT * huge
    op.close()


@pytest.mark.parametrize("depth", [10, 18, 20])  # meeting workgroups, and a finalize kernel
def test_captured_steps_replay(depth):
    """Two single steps captured on the caller's stream: every replay goes on
    with the dt chain, also between the handle's own runs."""
    import torch

    print("case:", depth, flush=True)
    mesh = host.mesh_uniform(depth)
    st = beach(mesh, 3)
    dt0 = host.initial_dt(mesh, st, COURANT) * 1e3
    ref = HostChain(mesh, st, dt0)
    op = operator(mesh)
    op.upload(*st)
    op.run(1, dt0, False)
    op.run(2, None, True, wait=False)  # a chain on the handle's own stream
    stream = torch.cuda.Stream()
    op.set_stream(stream.cuda_stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream, capture_error_mode="thread_local"):
        op.run(1, None, True, wait=False)
        op.run(1, None, False, wait=False)
    ref.run(3)
    for k in range(3):
        with torch.cuda.stream(stream):
            graph.replay()
        ref.run(2)
        n = (0, 8, 2)[k]
        op.run(n, None, True, wait=False)
        ref.run(n)
        assert op.run(0, None, True) == (ref.t, ref.dt)
        for a, b in zip(op.download(), ref.op.download()):
            assert np.array_equal(a, b)
    op.close()
    ref.op.close()


# around the length from which steps go into a graph (48, and 24 in each), from
# either buffer and direction
@pytest.mark.parametrize("depth", [6, 18, 19])
def test_long_runs_equal_single_traversals(depth):
    print("case:", depth, flush=True)
    mesh = host.mesh_uniform(depth)
    st = beach(mesh, 4)
    dt0 = host.initial_dt(mesh, st, COURANT) * 1e3
    ref = HostChain(mesh, st, dt0)
    op = operator(mesh, 128 if depth == 19 else None)
    op.upload(*st)
    fwd = False
    for i, n in enumerate([48, 49, 47, 74, 121]):
        got = op.run(n, dt0 if i == 0 else None, fwd)
        ref.run(n)
        fwd ^= n % 2 == 1
        assert got == (ref.t, ref.dt)
        for a, b in zip(op.download(), ref.op.download()):
            assert np.array_equal(a, b)
    op.close()
    ref.op.close()


def test_late_reductions():
    """On meshes of more than 4096 chunks a single step that nobody waits for
    leaves its partials to the remeshing after it, or to the next call that
    needs the slots: steps with and without remeshings between them, single
    traversals, longer runs and launch shapes against the host's chain."""
    print("case: depth 19, 128-cell chunks", flush=True)
    mesh = host.mesh_uniform(19)
    st = beach(mesh, 5)
    dt = host.initial_dt(mesh, st, COURANT) * 1e3
    ops = [swe.EulerTimestep(mesh, scaling=1e3, dry_tolerance=1e-3, courant=COURANT,
                             min_depth=18, max_depth=20, boundary=swe.BC_WALL)
           for _ in range(2)]
    for op in ops:
        op.set_tuning(128, 0)
        op.upload(*st)
    rng = np.random.default_rng(5)
    op, ref = ops
    t, fwd = 0.0, False

    def ref_steps(n, t, dt, fwd):
        for _ in range(n):
            res = ref.traverse(dt, fwd)
            t, dt, fwd = t + dt, COURANT * res.dt_cfl, not fwd
        return t, dt, fwd

    op.run(1, dt, fwd)
    t, dt, fwd = ref_steps(1, t, dt, fwd)
    for k in range(8):
        op.run(1, None, fwd, wait=False)
        half = 0.5 * dt
        t, dt, fwd = ref_steps(1, t, dt, fwd)
        if k == 1:  # the host's dt moves the state, not the device's chain
            assert op.traverse(half, fwd).dt_cfl == ref.traverse(half, fwd).dt_cfl
            fwd = not fwd
        if k in (2, 3, 6):  # a remeshing that changes the mesh, one that does not
            flags = np.zeros(op.n, np.int8)
            if k != 3:
                flags[rng.random(op.n) < 0.01] = 1
            assert op.adapt(flags)[0] == ref.adapt(flags)[0]
        if k == 4:
            op.run(3, None, fwd, wait=False)
            t, dt, fwd = ref_steps(3, t, dt, fwd)
        if k == 5:
            op.set_tuning(256, 0)
        if k != 0:
            assert op.run(0, None, fwd) == (t, dt), k
        for a, b in zip(op.download(), ref.download()):
            assert np.array_equal(a, b), k
    for o in ops:
        o.close()
