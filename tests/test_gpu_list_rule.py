"""Edge lists of a remeshed handle: the same steps before and after they are
stored, on every kind of call, and runs that do not wait for them."""
import numpy as np
import pytest
import torch

from samoa_amd import host, swe

pytestmark = pytest.mark.gpu

DT = 1e-3


def remeshed(depth, grow, chunk=256):
    """A remeshed handle and a new one on the same mesh (lists from the start)."""
    rng = np.random.default_rng(depth)
    mesh = host.mesh_uniform(depth)
    kw = dict(scaling=1000.0, dry_tolerance=1e-3, min_depth=max(depth - 2, 0), max_depth=depth + 2)
    old = swe.EulerTimestep(mesh, **kw)
    old.set_tuning(chunk, 0)
    b = -5.0 + 6.0 * rng.random(mesh.n)
    eta = np.maximum(0.2 * rng.normal(0, 1, mesh.n), b)
    h = eta - b
    old.upload(eta, h * rng.normal(0, 0.5, mesh.n), h * rng.normal(0, 0.5, mesh.n), b)
    old.adapt((rng.random(mesh.n) < 0.3).astype(np.int8) if grow
              else np.where(np.arange(mesh.n) < mesh.n // 2, -1, 0).astype(np.int8))
    new = swe.EulerTimestep(swe.Mesh(*old.download_mesh()), **kw)
    new.set_tuning(chunk, 0)
    new.upload(*old.download())
    return old, new


def same(old, new):
    for x, y in zip(old.download(), new.download()):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("chunk", [128, 256, 512])
@pytest.mark.parametrize("grow", [True, False])
@pytest.mark.parametrize("depth", [0, 6, 11])
def test_same_steps_across_the_storing(depth, grow, chunk):
    """Single steps until the lists are stored and beyond, then the adapted
    mesh again at once; device-pointer steps on another stream in between."""
    print("case:", depth, grow, chunk, flush=True)
    ops = remeshed(depth, grow, chunk)
    stream = torch.cuda.Stream()
    dt = [op.run(1, DT, True)[1] for op in ops]
    assert dt[0] == dt[1]
    for k in range(40):
        t = [op.run(1, None, k % 2 == 1) for op in ops]
        assert t[0] == t[1]
        if k in (0, 10, 23, 24, 25, 39):
            got = []
            for op in ops:
                q = [torch.as_tensor(a, device="cuda") for a in op.download()]
                out = [torch.empty_like(q[0]) for _ in range(3)]
                cfl = torch.zeros(1, dtype=torch.float64, device="cuda")
                torch.cuda.synchronize()
                op.step_device(*[a.data_ptr() for a in q + out], DT, True, cfl.data_ptr(),
                               stream=stream.cuda_stream)
                torch.cuda.synchronize()
                got.append(out + [cfl])
            assert all(torch.equal(x, y) for x, y in zip(*got))
    same(*ops)
    # a mesh after a long-lived one has its lists from its first step
    flags = (np.random.default_rng(1).random(ops[0].n) < 0.2).astype(np.int8)
    for op in ops:
        op.adapt(flags)
    for n in (1, 3, 60):
        t = [op.run(n, None, True) for op in ops]
        assert t[0] == t[1]
        same(*ops)
    for op in ops:
        op.close()


def test_a_run_on_a_remeshed_mesh_does_not_wait():
    """The lists are stored behind what is queued: runs that nobody waits for
    return while the stream still works on the caller's kernel."""
    old, new = remeshed(9, True)
    assert old.run(1, DT, True) == new.run(1, DT, True)
    stream = torch.cuda.Stream()
    old.set_stream(stream.cuda_stream)
    with torch.cuda.stream(stream):
        torch.cuda._sleep(int(2e8))  # a tenth of a second or more
        done = torch.cuda.Event()
        done.record(stream)
    for k in range(30):
        old.run(1, None, k % 2 == 0, wait=False)
    assert not done.query()
    for k in range(30):
        new.run(1, None, k % 2 == 0, wait=False)
    assert old.run(0, None, True) == new.run(0, None, True)
    same(old, new)
    old.close()
    new.close()
