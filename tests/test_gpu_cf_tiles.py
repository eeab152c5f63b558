"""Coarse/fine fills on boxes whose ghost slabs end at and just beyond the
fill's tile edges (32 parents along a face, 16 and 8 across) and on boxes of
two cells, with even and odd ghost widths (both children of a parent in the
slab, or one), against the oracle."""
import numpy as np
import pytest

import sledgehamr_amd as shm
from cases import real_scalar, rel_linf
from oracle_py import Oracle

pytestmark = pytest.mark.gpu

# Level-1 domain 96^3: 62 + 2 nghost cells are 33 parents and more; 34 and 18
# cells pass the 16- and 8-parent cuts; 2-cell edges; faces on the boundary.
BOXES = [[0, 0, 0, 61, 33, 17], [0, 40, 30, 17, 73, 31], [70, 4, 40, 71, 5, 95],
         [30, 50, 60, 33, 83, 93]]


def _pair(inp, prec, seed):
    sim, orc = shm.Simulation("RealScalar", inp, precision=prec), Oracle("RealScalar", inp)
    rng = np.random.default_rng(seed)
    for lev in (0, 1):
        if lev:
            sim.set_boxes(1, BOXES)
            orc.set_boxes(1, BOXES)
        for c in range(2):
            d = 0.3 * rng.standard_normal(sim.ncells(lev))
            sim.upload(lev, c, d)
            orc.upload(lev, c, d)
    return sim, orc


@pytest.mark.parametrize("interp", [0, 1, 2, 4])
@pytest.mark.parametrize("order", [1, 2, 3])
def test_rhs_at_slab_edges(order, interp):
    inp = real_scalar(N=48, order=order, nghost=order, L=48.0,
                      **{"amr.max_refinement_levels": 1, "amr.interpolation_type": interp,
                         "shm.allow_any_grid_size": 1})
    sim, orc = _pair(inp, shm.PREC_FP64, 3 + order)
    sim.fill_rhs(1, 0.0)
    orc.fill_rhs(1, 0.0)
    for c in range(2):
        # As the Rhs test of the plain layout: FP64 rounding of the stencil.
        assert rel_linf(sim.rhs(1, c), orc.rhs(1, c)) < 1e-13


@pytest.mark.parametrize("prec,tol", [(shm.PREC_FP64, 1e-12), (shm.PREC_FP32CS, 1e-6)])
@pytest.mark.parametrize("interp", [1, 2, 4])
@pytest.mark.parametrize("integrator,order", [(10, 2), (10, 3), (10, 1), (21, 3), (11, 2)])
def test_subcycled_steps(integrator, order, interp, prec, tol):
    """Steps whose stages read fills at the coarse level's old, new and
    intermediate times (two fine steps per coarse step)."""
    inp = real_scalar(N=48, order=order, nghost=order, L=48.0, cfl=0.2,
                      integrator=integrator,
                      **{"amr.max_refinement_levels": 1, "amr.interpolation_type": interp,
                         "shm.allow_any_grid_size": 1})
    sim, orc = _pair(inp, prec, 11)
    sim.evolve(2)
    orc.evolve(2)
    for lev in range(2):
        for c in range(2):
            assert rel_linf(sim.download(lev, c), orc.download(lev, c)) < tol, (lev, c)


@pytest.mark.parametrize("interp", [0, 1, 2, 4])
def test_whole_boxes(interp):
    inp = real_scalar(N=48, order=2, nghost=2, L=48.0,
                      **{"amr.max_refinement_levels": 1, "amr.interpolation_type": interp,
                         "shm.allow_any_grid_size": 1})
    sim, orc = _pair(inp, shm.PREC_FP64, 9)
    sim.fill_coarse_patch(1)
    orc.fill_coarse_patch(1)
    for c in range(2):
        assert rel_linf(sim.download(1, c), orc.download(1, c)) < 1e-13
