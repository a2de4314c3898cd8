"""NaN states in the toleranced step: its short solver leaves every edge with a
NaN to the general one, so the same cells set no CFL limit as in the exact step."""
import numpy as np
import pytest

from samoa_amd import host, swe

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solver", [swe.SOLVER_AUG_RIEMANN, swe.SOLVER_FWAVE])
@pytest.mark.parametrize("depth", [5, 9, 17])
def test_limits_beside_a_cell_without_numbers(depth, solver):
    """One cell's momentum is NaN, and its fast neighbours have the smallest
    limits of the mesh: they count in neither arithmetic.  (The cell is deeper
    than they are: a shallower one's edges have finite speeds in the general
    toleranced solver, whose square roots of NaN are 0.)"""
    print("case:", depth, solver, flush=True)
    mesh = host.mesh_uniform(depth)
    n = mesh.n
    ops = [swe.EulerTimestep(mesh, solver=solver, scaling=1e3, dry_tolerance=1e-3)
           for _ in range(2)]
    ops[1].set_arithmetic(swe.ARITH_TOLERANCED)
    rng = np.random.default_rng(depth)
    for cell in rng.integers(0, n, 6):
        near = [c for c in mesh.nbr.reshape(-1, 3)[cell] if c >= 0]
        eta, hu, hv, b = (0.01 * rng.normal(0, 1, n) for _ in range(4))
        b -= 5.0
        hu[near] = 12.0
        eta[cell], b[cell] = 0.1, -5.0
        whole = []
        for op in ops:
            op.upload(eta, hu, hv, b)
            whole.append(op.traverse(1e-6, True).dt_cfl)
        for bad in ("hu", "hv", "both"):
            u, v = hu.copy(), hv.copy()
            if bad != "hv":
                u[cell] = np.nan
            if bad != "hu":
                v[cell] = np.nan
            for fwd in (True, False):
                dt = []
                for op in ops:
                    op.upload(eta, u, v, b)
                    dt.append(op.traverse(1e-6, fwd).dt_cfl)
                # the neighbours' limits are gone, and nothing else is
                assert dt[0] > 1.001 * whole[0]
                assert abs(dt[1] - dt[0]) <= 1e-12 * dt[0]
    for op in ops:
        op.close()
