"""A level whose boxes tile the periodic domain is stored as one brick: steps,
tags, outputs, spectra and the finer level's ghost cells equal those of the
same domain in one box bit for bit, in the order of the boxes."""
import numpy as np
import pytest

import sledgehamr_amd as shm
from cases import complex_scalar, phase_transition, real_scalar

pytestmark = pytest.mark.gpu

ALLP = [shm.PREC_FP64, shm.PREC_FP32C, shm.PREC_FP32C16, shm.PREC_FP32CS]
ANY = {"shm.allow_any_grid_size": 1}


def _in_boxes(flat, N, boxes):
    u = flat.reshape(N, N, N)
    return np.concatenate([u[b[2]:b[5] + 1, b[1]:b[4] + 1, b[0]:b[3] + 1].ravel()
                           for b in np.asarray(boxes)])


def _pair(project, inp, prec, mg=None, boxes=None, seed=3):
    """The domain in one box, and in boxes (chopped, or an explicit list)."""
    one = shm.Simulation(project, inp, precision=prec)
    many = shm.Simulation(project, dict(inp, **({"amr.max_grid_size": mg} if mg else {})),
                          precision=prec)
    if boxes:
        many.set_boxes(0, boxes)
    bx = many.boxes(0)
    N = one.info["coarse_level_grid_size"]
    rng = np.random.default_rng(seed)
    for c in range(one.info["ncomp"]):
        d = 0.3 * rng.standard_normal(N ** 3) + (c == 0)
        one.upload(0, c, d)
        many.upload(0, c, _in_boxes(d, N, bx))
    return one, many, bx, N


def _same(one, many, bx, N, old=False):
    for c in range(one.info["ncomp"]):
        a = _in_boxes(one.download(0, c, old), N, bx)
        b = many.download(0, c, old)
        assert np.isfinite(a).all() and np.array_equal(a, b), c


# 6^3 boxes are smaller than a tile; 44 = 64 + 24 cells leave partial tiles.
@pytest.mark.parametrize("N,mg", [(12, 6), (32, 16), (64, 32), (88, 44), (96, 32)])
@pytest.mark.parametrize("prec", ALLP)
def test_steps(N, mg, prec):
    one, many, bx, N = _pair("ComplexScalar", complex_scalar(N=N, **ANY), prec, mg)
    for graphs in (False, True):
        for s in (one, many):
            s.set_graphs(graphs)
            s.advance(0, 3)
        _same(one, many, bx, N)
        _same(one, many, bx, N, old=True)
    assert many.get_launch(0)["fused"] == (1 if N >= 64 and prec != shm.PREC_FP32CS else 0)


SLABS = [[0, 0, 0, 31, 31, 9], [0, 0, 10, 31, 31, 31]]  # wrap along x and y
UNEVEN = [[0, 0, 0, 9, 31, 31], [10, 0, 0, 31, 15, 31], [10, 16, 0, 31, 31, 31]]


@pytest.mark.parametrize("boxes", [SLABS, UNEVEN])
@pytest.mark.parametrize("integrator", [10, 11, 21, 22])
def test_uneven_boxes(boxes, integrator):
    one, many, bx, N = _pair("RealScalar", real_scalar(N=32, order=3, integrator=integrator),
                             shm.PREC_FP32C16, boxes=boxes)
    for s in (one, many):
        s.advance(0, 3)
        s.fill_rhs(0, 0.1)
    _same(one, many, bx, N)
    for c in range(2):
        assert np.array_equal(_in_boxes(one.rhs(0, c), N, bx), many.rhs(0, c))


def test_boxes_that_leave_a_gap_stay_boxes():
    """Half the domain: not a tiling, so cells beside the gap keep ghosts."""
    sim = shm.Simulation("RealScalar", real_scalar(N=32), precision=shm.PREC_FP64)
    sim.set_boxes(0, [[0, 0, 0, 31, 31, 7], [0, 0, 8, 31, 31, 15]])
    sim.set_launch(fused=1)
    assert sim.get_launch(0)["fused"] == 0


@pytest.mark.parametrize("prec", [shm.PREC_FP64, shm.PREC_FP32C16])
def test_tags(prec):
    inp = complex_scalar(N=32, **{"amr.te_crit": 1e-3, "project.tag_strings": 1,
                                  "project.te_modifier": 1})
    one, many, bx, N = _pair("ComplexScalar", inp, prec, 16)
    for s in (one, many):
        s.advance(0, 1)
        s.create_shadow()
        s.advance(0, 1)
    (m0, c0, _), (m1, c1, _) = one.te_tag(0), many.te_tag(0)
    assert m0.any() and np.array_equal(_in_boxes(m0, N, bx), m1) and np.array_equal(c0, c1)


def test_outputs_and_spectra():
    one, many, bx, N = _pair("RealScalar", real_scalar(N=32, order=2, t_start=0.5),
                             shm.PREC_FP32C16, 8)
    for fn in range(3):
        for mode in (0, 1):
            (d0, n0), (d1, n1) = one.projection(fn, mode), many.projection(fn, mode)
            assert np.array_equal(n0, n1)
            # Sums arrive in atomic order: 32 terms, 32 eps each way.
            np.testing.assert_allclose(d0, d1, rtol=0, atol=64 * 2.3e-16 * np.abs(d0).max())
    one, many, bx, N = _pair("PhaseTransitionGW", phase_transition(N=32), shm.PREC_FP64, 16)
    for s in (one, many):
        s.advance(0, 2)
    _same(one, many, bx, N)
    b0, b1 = one.gw_spectrum(mode=1)[0], many.gw_spectrum(mode=1)[0]
    np.testing.assert_allclose(b0, b1, rtol=1e-12, atol=1e-15 * b0.max())


@pytest.mark.parametrize("interp", [1, 2, 4])
@pytest.mark.parametrize("integrator", [10, 21])
def test_finer_level_on_a_merged_base(integrator, interp):
    """Ghost cells of level 1 from coarse cells of several boxes and through
    the periodic boundary, and its average-down onto them."""
    inp = complex_scalar(N=32, integrator=integrator, L=8.0, nghost=3,
                         **{"amr.max_refinement_levels": 1, "amr.te_crit": 1e-3,
                            "amr.regrid_dt": 0.05, "amr.interpolation_type": interp})
    lev1 = [[20, 20, 20, 43, 43, 43], [0, 2, 0, 9, 13, 11], [44, 20, 20, 55, 31, 31]]
    one, many, bx, N = _pair("ComplexScalar", inp, shm.PREC_FP64, 16)
    rng = np.random.default_rng(8)
    for s in (one, many):
        s.set_boxes(1, lev1)
    for c in range(4):
        d = 0.3 * rng.standard_normal(one.ncells(1)) + (c == 0)
        one.upload(1, c, d)
        many.upload(1, c, d)
    for s in (one, many):
        s.evolve(4)
    _same(one, many, bx, N)
    for c in range(4):
        assert np.array_equal(one.download(1, c), many.download(1, c))
    assert one.events() == many.events()
