"""The adjoint kernel in one pass (meshes that do not fill the chip) and in two:
the same mesh alone and beside one that fills it, where every launch takes two
passes.  One chunk, two, the most in one pass (512 of 256 cells) and one more;
states whose edges are all clearly subcritical, none, and a beach's; NaN cells."""
import numpy as np
import pytest
import torch

from samoa_amd import host, swe

pytestmark = pytest.mark.gpu

FILL = 18


def state(kind, mesh, rng):
    n = mesh.n
    if kind == "ocean":
        return (0.1 * rng.normal(size=n), rng.normal(size=n), rng.normal(size=n),
                -100.0 + rng.normal(size=n))
    cen = mesh.centroids()
    if kind == "beach":
        b = -8.0 + 11.0 * cen[:, 0] + 0.5 * np.sin(9.0 * cen[:, 1])
        eta = np.where(np.hypot(cen[:, 0] - 0.3, cen[:, 1] - 0.5) < 0.2, 1.5, 0.0)
    else:
        b = -1.0 + 0.3 * rng.normal(size=n)
        eta = b + np.abs(rng.normal(size=n)) * (rng.random(n) < 0.7)
    h = np.maximum(eta - b, 0.0)
    eta = np.where(h > 1e-3, eta, np.minimum(b, 0.0))
    h = np.where(h > 1e-3, h, 0.0)
    hu, hv = (h * rng.normal(size=n) * (6.0 if kind == "fast" else 2.0) for _ in range(2))
    if kind == "holes":
        hu[rng.random(n) < 0.01] = np.nan
    return eta, hu, hv, b


@pytest.mark.parametrize("depth,extra", [(0, False), (6, False), (7, False), (8, False),
                                         (11, False), (16, False), (16, True)])
@pytest.mark.parametrize("solver", [swe.SOLVER_AUG_RIEMANN, swe.SOLVER_FWAVE])
def test_one_pass_and_two(depth, extra, solver):
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
    full = host.mesh_uniform(FILL)
    kw = dict(scaling=1e3, dry_tolerance=1e-3, solver=solver, boundary=swe.BC_WALL)
    alone = swe.EulerTimestep(mesh, **kw)
    beside = swe.Batch([mesh, full], [kw, kw])
    n, total = mesh.n, mesh.n + full.n
    dev = lambda x: torch.tensor(x, device="cuda")  # noqa: E731
    p = lambda ts: [t.data_ptr() for t in ts]  # noqa: E731
    dt = torch.full((2,), 1e-3, dtype=torch.float64, device="cuda")
    calm = np.zeros(full.n), np.full(full.n, -100.0)
    for kind in ("ocean", "beach", "fast", "holes"):
        print("case:", depth, extra, solver, kind, flush=True)
        rng = np.random.default_rng(depth)
        st = state(kind, mesh, rng)
        q = [dev(np.concatenate([a, calm[1] if k == 3 else calm[0]])) for k, a in enumerate(st)]
        lam = [torch.tensor(rng.normal(size=total), device="cuda") for _ in range(3)]
        for forward in (True, False):
            masks = torch.zeros(total, dtype=torch.int8, device="cuda")
            mid = [torch.empty_like(q[0]) for _ in range(3)]
            want = [torch.empty_like(q[0]) for _ in range(3)] + [torch.zeros_like(q[0])]
            torch.cuda.synchronize()
            beside.forward_device(*p(q + mid), dt.data_ptr(), forward, masks=masks.data_ptr())
            beside.adjoint_device(*p(q), masks.data_ptr(), *p(lam), *p(want), dt.data_ptr(),
                                  forward)
            torch.cuda.synchronize()
            for chunk in (128, 256, 512):
                alone.set_tuning(chunk, 0)
                got = [torch.empty(n, dtype=torch.float64, device="cuda") for _ in range(3)]
                got.append(torch.zeros_like(got[0]))
                torch.cuda.synchronize()
                alone.adjoint_device(*p([a[:n] for a in q]), masks.data_ptr(),
                                     *p([a[:n] for a in lam]), *p(got), dt.data_ptr(), forward)
                torch.cuda.synchronize()
                for a, w in zip(got, want):
                    a, w = a.cpu().numpy(), w[:n].cpu().numpy()
                    assert kind == "holes" or np.isfinite(a).all()
                    assert np.array_equal(a, w, equal_nan=True), (kind, chunk, forward)
    alone.close()
    beside.close()
