"""Calls that a caller captured, replayed while the handle's own runs are going
on: the dt chain that a run leaves for the next one stands, and a captured run
takes it up."""
import numpy as np
import pytest
import torch

from samoa_amd import host, swe

pytestmark = pytest.mark.gpu

COURANT = 0.45


def setup(depth):
    mesh = host.mesh_uniform(depth)
    rng = np.random.default_rng(depth)
    b = -5.0 + 0.1 * rng.normal(0, 1, mesh.n)
    st = [0.1 * rng.normal(0, 1, mesh.n) for _ in range(3)] + [b]
    op = swe.EulerTimestep(mesh, scaling=1e3, dry_tolerance=1e-3, courant=COURANT)
    op.upload(*st)
    return mesh, st, op, COURANT * op.traverse(1e-6, True).dt_cfl


def plain(depth, parts):
    """(time, dt) after each part of a run, without anything else going on."""
    _, st, op, dt0 = setup(depth)
    op.upload(*st)
    got, fwd = [], True
    for k, n in enumerate(parts):
        got.append(op.run(n, dt0 if k == 0 else None, fwd, time=0.0))
        fwd = fwd if n % 2 == 0 else not fwd
    state = op.download()
    op.close()
    return got, state


# meshes whose runs are a chain, whose workgroups meet, and with a finalize kernel
@pytest.mark.parametrize("depth", [10, 18, 20])
@pytest.mark.parametrize("cfl", [True, False])
def test_replayed_traversals_between_runs(depth, cfl):
    """A traversal of other, faster states (device pointers) is captured once
    and replayed after each of the handle's runs that nobody waited for."""
    print("case:", depth, cfl, flush=True)
    parts = [1, 1, 2, 1, 3]
    want, state = plain(depth, parts)
    mesh, st, op, dt0 = setup(depth)
    op.upload(*st)
    stream = torch.cuda.Stream()
    fast = [torch.as_tensor(a, device="cuda") for a in st]
    fast[1] = fast[1] + 30.0
    out = [torch.empty_like(a) for a in fast[:3]]
    dt = torch.full((1,), 1e-6, dtype=torch.float64, device="cuda")
    lim = torch.zeros_like(dt)
    p = lambda ts: [t.data_ptr() for t in ts]  # noqa: E731
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream, capture_error_mode="thread_local"):
        op.forward_device(*p(fast), *p(out), dt.data_ptr(), True,
                          dt_cfl=lim.data_ptr() if cfl else 0, stream=stream.cuda_stream)
    fwd = True
    for k, n in enumerate(parts):
        if k == 0:
            op.run(n, dt0, fwd, time=0.0)
        else:
            op.run(n, None, fwd, wait=False)
        fwd = fwd if n % 2 == 0 else not fwd
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            graph.replay()
        torch.cuda.synchronize()
        if k in (1, 4):
            assert op.run(0, None, fwd) == want[k]
    for x, y in zip(op.download(), state):
        assert np.array_equal(x, y)
    op.close()


@pytest.mark.parametrize("depth", [10, 18, 20])
def test_replayed_steps_after_runs_on_the_own_stream(depth):
    """Two single steps captured on a caller's stream; the handle goes back to
    its own, and replays take turns with runs there that nobody waited for."""
    print("case:", depth, flush=True)
    parts = [1, 2, 2, 2, 2, 6, 2]
    want, state = plain(depth, parts)
    _, st, op, dt0 = setup(depth)
    op.upload(*st)
    stream = torch.cuda.Stream()
    op.set_stream(stream.cuda_stream)
    op.run(1, dt0, True, time=0.0)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream, capture_error_mode="thread_local"):
        op.run(1, None, False, wait=False)
        op.run(1, None, True, wait=False)
    op.set_stream(0)
    for k, n in enumerate(parts[1:], 1):
        if k % 2:
            op.run(n, None, False, wait=False)
        else:
            torch.cuda.synchronize()
            with torch.cuda.stream(stream):
                graph.replay()
            torch.cuda.synchronize()
        if k in (3, 4, 6):
            assert op.run(0, None, False) == want[k]
    for x, y in zip(op.download(), state):
        assert np.array_equal(x, y)
    op.close()
