"""The name of the device's null stream, SWE_STREAM_NULL, where it is not a
handle's launch argument: calls without a handle take it as NULL, and a handle
does not launch on it."""
import ctypes as C

import numpy as np
import pytest
import torch

from samoa_amd import _native, host, swe

pytestmark = pytest.mark.gpu


def test_handles_refuse_it():
    mesh = host.mesh_uniform(6)
    z = np.zeros(mesh.n)
    with swe.EulerTimestep(mesh) as op:
        op.upload(z, z, z, z - 1.0)
        want = op.run(2, 1e-3, True)
        with pytest.raises(_native.SweError):
            op.set_stream(swe.STREAM_NULL)
        op.upload(z, z, z, z - 1.0)
        assert op.stream == 0 and op.run(2, 1e-3, True) == want
    batch = swe.Batch([mesh], [{}])
    with pytest.raises(_native.SweError):
        batch.set_stream(swe.STREAM_NULL)
    batch.close()


def test_calls_without_a_handle_take_it():
    mesh = host.mesh_uniform(9)
    rng = np.random.default_rng(0)
    dev = lambda a: torch.as_tensor(np.ascontiguousarray(a), device="cuda")  # noqa: E731
    p = lambda ts: [t.data_ptr() for t in ts]  # noqa: E731
    lib = _native.load()
    q = [dev(0.1 * rng.normal(size=mesh.n)) for _ in range(3)] + [dev(np.full(mesh.n, -5.0))]
    topo = [dev(mesh.depth.astype(np.int8)), dev(mesh.plotter.astype(np.int8)),
            dev(np.asarray(mesh.nbr, np.int32).reshape(-1))]
    dm = _native.DeviceMesh(n_cells=mesh.n, depth=topo[0].data_ptr(), plotter=topo[1].data_ptr(),
                            nbr=topo[2].data_ptr(), scaling=1e3, g=swe.G, dry_tolerance=1e-3,
                            min_depth=0, max_depth=12, solver=0, boundary=0)
    n = mesh.n  # a remeshing that splits every cell in two
    code = torch.full((n,), 4, dtype=torch.int8, device="cuda")
    base = 2 * torch.arange(n, dtype=torch.int64, device="cuda")
    new = [dev(rng.normal(size=2 * n)) for _ in range(4)]
    got = []
    for stream in (None, swe.STREAM_NULL):
        out = [torch.zeros_like(q[0]) for _ in range(3)]
        cfl = torch.zeros(1, dtype=torch.float64, device="cuda")
        _native.check("noalloc", lib.swe_step_device_noalloc(
            C.byref(dm), *p(q + out), 1e-3, 1, cfl.data_ptr(), None, None, stream))
        back = [torch.zeros_like(q[0]) for _ in range(4)]
        _native.check("transfer", lib.swe_transfer_adjoint_device(
            n, code.data_ptr(), base.data_ptr(), 0, *p(new), *p(back), stream))
        got.append(out + [cfl] + back)
    torch.cuda.synchronize()
    assert all(torch.equal(x, y) for x, y in zip(*got))
    assert float(got[0][3]) > 0.0 and float(got[0][4].abs().max()) > 0.0
