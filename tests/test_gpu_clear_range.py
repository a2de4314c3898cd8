"""Momenta and beds over the whole range of doubles, zeros and equal neighbours
among them, against the oracle bit for bit: the shortcut solver's shared
reciprocals round correctly wherever its test lets a cell through, and the
cells at the ends of its range take the general path."""
import numpy as np
import pytest

import pyoracle as po
from samoa_amd import swe

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solver", [swe.SOLVER_AUG_RIEMANN, swe.SOLVER_FWAVE])
@pytest.mark.parametrize("lowest", [-320, -250, -222, -216, -110, -95, -30])
def test_step_equals_the_oracle(solver, lowest):
    d = 9
    plotter, co, nbr = po.mesh_uniform(d)
    mesh = swe.Mesh(np.full(plotter.shape[0], d, np.int8), plotter, nbr, co)
    n = mesh.n
    rng = np.random.default_rng(-lowest)
    tiny = lambda top: (rng.choice([-1.0, 1.0], n) * 10.0 ** rng.uniform(lowest, top, n) *  # noqa: E731
                        (rng.random(n) < 0.8))
    patch = np.arange(n) // 8  # cells of a patch share their bed, most their surface
    flat = rng.random(n)[patch]
    b = np.where(flat < 0.4, -3.0 - flat, np.where(flat < 0.7, -3.0 + tiny(-3), tiny(-1)))
    eta = np.where(flat < 0.7, 0.0, 3.0) + np.where(rng.random(n) < 0.4, tiny(-1), 0.0)
    hu, hv = tiny(0), tiny(0)
    op = swe.EulerTimestep(mesh, scaling=100.0, dry_tolerance=1e-3, solver=solver)
    ref = [eta, hu, hv, b]
    op.upload(*ref)
    for fwd in (True, False, True):
        res = op.traverse(0.05, fwd)
        e, u, v, _, cand, _ = po.step(mesh.depth, mesh.plotter, mesh.nbr, ref, 0.05, scaling=100.0,
                                      drytol=1e-3, dmin=d, dmax=d, bc=swe.BC_OUTFLOW,
                                      solver=solver, forward=fwd)
        ref = [e, u, v, b]
        assert res.dt_cfl == cand
        for x, y in zip(op.download(), ref):
            assert np.array_equal(x, y)
    op.close()
