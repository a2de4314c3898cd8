"""Bathymetry of split cells averaged over every number of halvings at which
the device changes how it samples (in the emit, by a wave, by a wave with
serial parts), bit-identical to the host's average on the new mesh."""
import numpy as np
import pytest

from samoa_amd import bathymetry as bt
from samoa_amd import host, swe

pytestmark = pytest.mark.gpu

NODES = 257  # on the unit square: data depth 16


@pytest.mark.parametrize("levels", [0, 1, 2, 3, 5, 6, 7, 8, 12, 15])
@pytest.mark.parametrize("shallow", [False, True])
def test_split_cells_average_the_raster(levels, shallow):
    """Children of depth d + 1 take `levels` halvings, those split again one
    fewer.  shallow: every cell is above the run's minimum depth, so the
    emit samples all children itself."""
    cap = min(19, 5 + levels)
    d, dmax = cap - levels - 1, cap - 3
    if dmax <= d:  # the depth limits of the run end above the children
        d, dmax = d, d + 2
    rng = np.random.default_rng(levels)
    values = rng.normal(-50.0, 30.0, (NODES, NODES))
    r = bt.Raster(values, 0.0, 0.0, 1.0 / (NODES - 1), 1.0 / (NODES - 1))
    mesh = host.mesh_uniform(d)
    b = bt.cell_bathymetry(r, mesh.coords, 1.0, (0.0, 0.0), depth=mesh.depth, dmax=dmax)
    z = np.zeros(mesh.n)
    print("case: levels", levels, "depth", d, "dmax", dmax, "shallow", shallow, flush=True)
    op = swe.EulerTimestep(mesh, dry_tolerance=1e-3, min_depth=18 if shallow else 0,
                           max_depth=dmax)
    op.upload(z, z, z, b)
    op.set_bathymetry_raster(r.values, r.x0, r.y0, r.dx, r.dy, (0.0, 0.0))
    flags = (rng.random(mesh.n) < 0.4).astype(np.int8)
    flags[:2] = 1
    n, _ = op.adapt(flags)
    assert n > mesh.n
    depth = op.download_mesh()[0]
    coords = host.coords_from_depths(depth)[1]
    want = bt.cell_bathymetry(r, coords, 1.0, (0.0, 0.0), depth=depth, dmax=dmax)
    assert np.array_equal(op.download()[3], want)
    op.close()
