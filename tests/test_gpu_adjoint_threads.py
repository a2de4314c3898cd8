"""The adjoint kernel with one and two threads per cell (meshes of few chunks):
one cell pair, part of a chunk, the most chunks with two threads (256 of 256
cells, 512 of 128) and one more.  Its results do not depend on the chunks, so
every chunk size gives those of 512-cell chunks, which have one thread per cell."""
import numpy as np
import pytest
import torch

from samoa_amd import host, swe

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("depth,extra", [(0, False), (5, False), (9, False), (15, False),
                                         (15, True)])
@pytest.mark.parametrize("solver", [swe.SOLVER_AUG_RIEMANN, swe.SOLVER_FWAVE])
def test_threads_per_cell(depth, extra, solver):
    print("case:", depth, extra, solver, flush=True)
    mesh = host.mesh_uniform(depth)
    if extra:
        with swe.EulerTimestep(mesh, min_depth=depth, max_depth=depth + 1) as op:
            z = np.zeros(mesh.n)
            op.upload(z, z, z, z)
            flags = np.zeros(mesh.n, np.int8)
            flags[12345] = 1
            op.adapt(flags)
            d, p, nbr = op.download_mesh()
        mesh = swe.Mesh(d, p, nbr, host.coords_from_depths(d)[1])
    rng = np.random.default_rng(depth)
    cen = mesh.centroids()
    b = -8.0 + 11.0 * cen[:, 0] + 0.5 * np.sin(9.0 * cen[:, 1])
    eta = np.where(np.hypot(cen[:, 0] - 0.3, cen[:, 1] - 0.5) < 0.2, 1.5, 0.0)
    wet = eta > b + 1e-3
    eta = np.where(wet, eta, np.minimum(b, 0.0))
    # slow over most of the mesh, fast in places
    hu, hv = (np.where(wet, rng.normal(size=mesh.n) * (0.1 + 20.0 * (rng.random(mesh.n) < 0.02)),
                       0.0) for _ in range(2))
    dev = lambda x: torch.tensor(x, device="cuda")  # noqa: E731
    q = [dev(x) for x in (eta, hu, hv, b)]
    lam = [dev(rng.normal(size=mesh.n)) for _ in range(3)]
    dt = torch.full((1,), 1e-3, dtype=torch.float64, device="cuda")
    masks = torch.zeros(mesh.n, dtype=torch.int8, device="cuda")
    op = swe.EulerTimestep(mesh, scaling=1e3, dry_tolerance=1e-3, solver=solver,
                           boundary=swe.BC_WALL)
    for forward in (True, False):
        want = None
        for chunk in (512, 256, 128):
            op.set_tuning(chunk, 0)
            out = [torch.empty_like(q[0]) for _ in range(3)]
            gb = torch.zeros_like(q[0])
            torch.cuda.synchronize()
            op.forward_device(*[x.data_ptr() for x in q + out], dt.data_ptr(), forward,
                              masks=masks.data_ptr())
            op.adjoint_device(*[x.data_ptr() for x in q], masks.data_ptr(),
                              *[x.data_ptr() for x in lam + out], gb.data_ptr(), dt.data_ptr(),
                              forward)
            torch.cuda.synchronize()
            got = [x.cpu().numpy() for x in out + [gb]]
            if want is None:
                want = got
                assert all(np.isfinite(x).all() for x in got)
            for a, w in zip(got, want):
                assert np.array_equal(a, w), chunk
    op.close()
