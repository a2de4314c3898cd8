"""The device-pointer entry points on each stream a caller can name: the
handle's own, the device's null stream, and one of the caller's, with the
caller's work before and after on torch's matching stream."""
import numpy as np
import pytest
import torch

from samoa_amd import host, swe
from samoa_amd.adjoint import GaugeInversion

pytestmark = pytest.mark.gpu


def chain(kind, depth, solver):
    """Two traversals and the reverse of the first, torch's work in between."""
    mesh = host.mesh_uniform(depth)
    rng = np.random.default_rng(depth)
    side = torch.cuda.Stream() if kind == "side" else torch.cuda.current_stream()
    name = {"own": 0, "null": swe.STREAM_NULL, "side": side.cuda_stream}[kind]
    op = swe.EulerTimestep(mesh, solver=solver)
    with torch.cuda.stream(side):
        dev = lambda a: torch.as_tensor(a, dtype=torch.float64, device="cuda")  # noqa: E731
        b = dev(-2.0 + 0.1 * rng.normal(0, 1, mesh.n))
        q = [dev(0.01 * rng.normal(0, 1, mesh.n)) for _ in range(3)]
        p = lambda ts: [t.data_ptr() for t in ts]  # noqa: E731
        mid, out, lam = ([torch.empty_like(b) for _ in range(3)] for _ in range(3))
        masks = torch.empty(mesh.n, dtype=torch.int8, device="cuda")
        dt = torch.full((1,), 1e-5, dtype=torch.float64, device="cuda")
        cfl, gb = torch.zeros_like(dt), torch.zeros_like(b)
        for _ in range(3):
            op.forward_device(*p(q), b.data_ptr(), *p(mid), dt.data_ptr(), True,
                              dt_cfl=cfl.data_ptr(), masks=masks.data_ptr(), stream=name)
            mid2 = [2.0 * m for m in mid]
            op.step_device(*p(mid2), b.data_ptr(), *p(out), 1e-5, False, cfl.data_ptr(),
                           stream=name)
            seeds = [o + 1.0 for o in out]
            op.adjoint_device(*p(q), b.data_ptr(), masks.data_ptr(), *p(seeds), *p(lam),
                              gb.data_ptr(), dt.data_ptr(), True, stream=name)
            q = [x + 1e-3 * y for x, y in zip(q, lam)]
        got = torch.stack(q + out + [gb, masks.double(), cfl.expand(mesh.n)])
    torch.cuda.synchronize()
    op.close()
    return got


@pytest.mark.parametrize("solver", [swe.SOLVER_AUG_RIEMANN, swe.SOLVER_FWAVE])
@pytest.mark.parametrize("depth", [3, 10, 15])
def test_same_results_on_every_stream(depth, solver):
    want = chain("own", depth, solver)
    for kind in ("null", "side"):
        assert torch.equal(want, chain(kind, depth, solver)), kind


@pytest.mark.parametrize("steps", [1, 2, 9])
def test_gathered_series_equal_the_checkpointed_sweep(steps):
    """One gather over the kept elevations against one per step, with gauges
    that repeat and lie at both ends."""
    mesh = host.mesh_uniform(9)
    eta, _, _, b = host.tsunami(mesh, seed=4, drytol=1e-3)
    gauges = np.array([0, 7, mesh.n - 1, 7])
    got = []
    for every in ("all", 2):
        prob = GaugeInversion(mesh, gauges, steps, dict(scaling=1.0e6, dry_tolerance=1e-3),
                              checkpoint_every=every)
        e, bed = (torch.tensor(a, device="cuda", requires_grad=True) for a in (eta, b))
        prob.record_dt(e, bed, 1.0)
        series = prob.gauge_series(e, bed)
        (series ** 2).sum().backward()
        got.append((series.detach(), e.grad, bed.grad))
        prob.close()
    assert got[0][0].shape == (steps, 4)
    assert torch.equal(got[0][0], got[1][0])
    for x, y in zip(*(g[1:] for g in got)):
        # two gauges on one cell are added in either order
        assert torch.allclose(x, y, rtol=1e-12, atol=1e-12 * float(x.abs().max()))
