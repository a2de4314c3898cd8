"""NaN states and the CFL minimum.  A cell whose speeds are NaN sets no limit,
however a launch's workgroups reduce their partials: here every cell of a
chunk is NaN, or of the mesh.  The limit comes from one fast cell elsewhere, so
it is the one of the state without NaN."""
import numpy as np
import pytest

from samoa_amd import host, swe

pytestmark = pytest.mark.gpu

COURANT, DT = 0.45, 1e-6
HUGE = np.finfo(float).max


def still_water(n, fast):
    """Still water 5 m deep, with 200 m/s in cell `fast`: far above the
    14 m/s at which water runs out beside a cell without numbers."""
    eta, hu, hv, b = np.zeros(n), np.zeros(n), np.zeros(n), np.full(n, -5.0)
    hu[fast] = 1000.0
    return [eta, hu, hv, b]


# one thread per cell in a chain of chunks of 512; 1024 chunks: the single step
# meets, the run is a chain; 2048: both meet; 8192: a finalize kernel
@pytest.mark.parametrize("depth,chunk", [(9, 256), (9, 512), (17, 256), (18, 256), (18, 512),
                                         (20, 256)])
@pytest.mark.parametrize("arithmetic", [swe.ARITH_EXACT, swe.ARITH_TOLERANCED])
def test_a_chunk_without_numbers(depth, chunk, arithmetic):
    print("case:", depth, chunk, arithmetic, flush=True)
    mesh = host.mesh_uniform(depth)
    n = mesh.n
    op = swe.EulerTimestep(mesh, scaling=1e3, dry_tolerance=1e-3, courant=COURANT)
    op.set_tuning(chunk, 0)
    op.set_arithmetic(arithmetic)
    q = still_water(n, n // 3)
    op.upload(*q)
    whole = op.traverse(DT, True).dt_cfl
    op.upload(*q)
    run = op.run(3, DT, True)
    assert 0.0 < whole < HUGE and 0.0 < run[1] < HUGE
    for first in (0, (2 * n // 3) // chunk * chunk, n - chunk):
        if first <= n // 3 < first + chunk:
            continue
        for k in range(3):
            bad = [a.copy() for a in q]
            bad[k][first:first + chunk] = np.nan
            op.upload(*bad)
            assert op.traverse(DT, True).dt_cfl == whole
            op.upload(*bad)
            assert op.run(3, DT, True) == run
            after = op.download()[0]
            assert np.isfinite(after[n // 3])
    for k in range(3):
        bad = [a.copy() for a in q]
        bad[k][:] = np.nan
        op.upload(*bad)
        assert op.traverse(DT, True).dt_cfl == HUGE
        op.upload(*bad)
        assert op.run(3, DT, True)[1] == COURANT * HUGE
    op.close()


@pytest.mark.parametrize("depth", [17, 18])
def test_the_forms_that_meet_on_a_callers_stream(depth):
    """Device-pointer steps, and short and captured runs on a caller's stream."""
    import torch

    print("case:", depth, flush=True)
    mesh = host.mesh_uniform(depth)
    n = mesh.n
    op = swe.EulerTimestep(mesh, scaling=1e3, dry_tolerance=1e-3, courant=COURANT)
    q = still_water(n, n // 3)
    op.upload(*q)
    want = [op.run(1, DT, True)[1], None]
    want[1] = op.run(1, None, False)[1]
    bad = [a.copy() for a in q]
    bad[1][:256] = np.nan
    dev = [torch.as_tensor(a, device="cuda") for a in bad]
    out = [torch.empty_like(a) for a in dev[:3]]
    cfl = torch.zeros(1, dtype=torch.float64, device="cuda")
    p = lambda ts: [t.data_ptr() for t in ts]  # noqa: E731
    op.step_device(*p(dev), *p(out), DT, True, cfl.data_ptr(), stream=swe.STREAM_NULL)
    assert COURANT * float(cfl) == want[0]
    stream = torch.cuda.Stream()
    op.set_stream(stream.cuda_stream)
    op.upload(*bad)
    assert op.run(1, DT, True)[1] == want[0]
    assert op.run(1, None, False)[1] == want[1]
    op.upload(*bad)
    op.run(1, DT, True)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream, capture_error_mode="thread_local"):
        op.run(1, None, False, wait=False)
        op.run(1, None, True, wait=False)
    for _ in range(2):
        with torch.cuda.stream(stream):
            graph.replay()
        got = op.run(0, None, True)
        assert 0.0 < got[1] < HUGE and np.isfinite(got[0])
    op.close()
