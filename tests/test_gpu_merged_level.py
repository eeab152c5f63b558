"""A level whose boxes tile the periodic domain, stored as one brick or
(shm.merge_boxes = 0, and always over 4 GiB per FP64 component) box by box with
ghost copies: steps, tags, outputs, spectra and the finer level's ghost cells
equal those of the same domain in one box bit for bit, in the order of the
boxes, and the oracle's, which steps box by box."""
import numpy as np
import pytest

import sledgehamr_amd as shm
from cases import complex_scalar, phase_transition, real_scalar, rel_linf
from oracle_py import Oracle

pytestmark = pytest.mark.gpu

ALLP = [shm.PREC_FP64, shm.PREC_FP32C, shm.PREC_FP32C16, shm.PREC_FP32CS]
ANY = {"shm.allow_any_grid_size": 1}


def _in_boxes(flat, N, boxes):
    u = flat.reshape(N, N, N)
    return np.concatenate([u[b[2]:b[5] + 1, b[1]:b[4] + 1, b[0]:b[3] + 1].ravel()
                           for b in np.asarray(boxes)])


def _pair(project, inp, prec, mg=None, boxes=None, seed=3, merge=1):
    """The domain in one box, and in boxes (chopped, or an explicit list)."""
    one = shm.Simulation(project, inp, precision=prec)
    many = shm.Simulation(project, dict(inp, **{"shm.merge_boxes": merge},
                                        **({"amr.max_grid_size": mg} if mg else {})),
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


MERGE = pytest.mark.parametrize("merge", [1, 0])


# 6^3 boxes are smaller than a tile; 88 = 64 + 24 cells leave partial tiles.
@MERGE
@pytest.mark.parametrize("N,mg", [(12, 6), (32, 16), (64, 32), (88, 44), (96, 32)])
@pytest.mark.parametrize("prec", ALLP)
def test_steps(N, mg, prec, merge):
    one, many, bx, N = _pair("ComplexScalar", complex_scalar(N=N, **ANY), prec, mg, merge=merge)
    for graphs in (False, True):
        for s in (one, many):
            s.set_graphs(graphs)
            s.advance(0, 3)
        _same(one, many, bx, N)
        _same(one, many, bx, N, old=True)
    assert many.get_launch(0)["fused"] == \
        (1 if merge and N >= 64 and prec != shm.PREC_FP32CS else 0)


SLABS = [[0, 0, 0, 31, 31, 9], [0, 0, 10, 31, 31, 31]]  # wrap along x and y
UNEVEN = [[0, 0, 0, 9, 31, 31], [10, 0, 0, 31, 15, 31], [10, 16, 0, 31, 31, 31]]


@MERGE
@pytest.mark.parametrize("boxes", [SLABS, UNEVEN])
@pytest.mark.parametrize("integrator", [10, 11, 21, 22])
def test_uneven_boxes(boxes, integrator, merge):
    one, many, bx, N = _pair("RealScalar", real_scalar(N=32, order=3, integrator=integrator),
                             shm.PREC_FP32C16, boxes=boxes, merge=merge)
    for s in (one, many):
        s.advance(0, 3)
        s.fill_rhs(0, 0.1)
    _same(one, many, bx, N)
    for c in range(2):
        assert np.array_equal(_in_boxes(one.rhs(0, c), N, bx), many.rhs(0, c))


@MERGE
@pytest.mark.parametrize("integrator", [10, 11, 21])
@pytest.mark.parametrize("boxes", [SLABS, UNEVEN, None])
def test_against_oracle(boxes, integrator, merge):
    """FP64, rounding of three steps (as the other parity tests take it)."""
    inp = real_scalar(N=32, order=2, integrator=integrator, L=32.0)
    one, many, bx, N = _pair("RealScalar", inp, shm.PREC_FP64, 16 if boxes is None else None,
                             boxes=boxes, merge=merge)
    orc = Oracle("RealScalar", dict(inp, **({"amr.max_grid_size": 16} if boxes is None else {})))
    if boxes:
        orc.set_boxes(0, boxes)
    for c in range(2):
        orc.upload(0, c, many.download(0, c))
    many.advance(0, 3)
    orc.advance(0, 3)
    for c in range(2):
        assert rel_linf(many.download(0, c), orc.download(0, c)) < 1e-12, c


@MERGE
@pytest.mark.parametrize("integrator", [10, 21, 22])
@pytest.mark.parametrize("prec", [shm.PREC_FP64, shm.PREC_FP32C16, shm.PREC_FP32CS])
def test_gw_steps(prec, integrator, merge):
    """Fourteen components in three groups; box by box, every stage state that
    a stage stores for the next one is copied between boxes."""
    one, many, bx, N = _pair("PhaseTransitionGW", phase_transition(N=32, integrator=integrator),
                             prec, 16, merge=merge)
    for s in (one, many):
        s.advance(0, 2)
    _same(one, many, bx, N)


def test_boxes_that_leave_a_gap_stay_boxes():
    """Half the domain: not a tiling, so cells beside the gap keep ghosts.
    Three RKN4 steps at radius 1 reach 9 planes; planes further from the gap
    hold what they hold on the whole domain."""
    one = shm.Simulation("RealScalar", real_scalar(N=32), precision=shm.PREC_FP64)
    sim = shm.Simulation("RealScalar", real_scalar(N=32), precision=shm.PREC_FP64)
    boxes = [[0, 0, 0, 31, 31, 11], [0, 0, 12, 31, 31, 27]]
    sim.set_boxes(0, boxes)
    sim.set_launch(fused=1)
    assert sim.get_launch(0)["fused"] == 0
    rng = np.random.default_rng(6)
    for c in range(2):
        d = 0.3 * rng.standard_normal(32 ** 3)
        one.upload(0, c, d)
        sim.upload(0, c, _in_boxes(d, 32, boxes))
    for s in (one, sim):
        s.advance(0, 3)
    for c in range(2):
        a = one.download(0, c).reshape(32, 32, 32)[9:19]
        b = sim.download(0, c).reshape(28, 32, 32)[9:19]
        assert np.isfinite(a).all() and np.array_equal(a, b), c


@MERGE
@pytest.mark.parametrize("prec", [shm.PREC_FP64, shm.PREC_FP32C16])
def test_tags(prec, merge):
    inp = complex_scalar(N=32, **{"amr.te_crit": 1e-3, "project.tag_strings": 1,
                                  "project.te_modifier": 1})
    one, many, bx, N = _pair("ComplexScalar", inp, prec, 16, merge=merge)
    for s in (one, many):
        s.advance(0, 1)
        s.create_shadow()
        s.advance(0, 1)
    (m0, c0, _), (m1, c1, _) = one.te_tag(0), many.te_tag(0)
    assert m0.any() and np.array_equal(_in_boxes(m0, N, bx), m1) and np.array_equal(c0, c1)


@MERGE
def test_outputs_and_spectra(merge):
    one, many, bx, N = _pair("RealScalar", real_scalar(N=32, order=2, t_start=0.5),
                             shm.PREC_FP32C16, 8, merge=merge)
    for fn in range(3):
        for mode in (0, 1):
            (d0, n0), (d1, n1) = one.projection(fn, mode), many.projection(fn, mode)
            assert np.array_equal(n0, n1)
            # Sums arrive in atomic order: 32 terms, 32 eps each way.
            np.testing.assert_allclose(d0, d1, rtol=0, atol=64 * 2.3e-16 * np.abs(d0).max())
    one, many, bx, N = _pair("PhaseTransitionGW", phase_transition(N=32), shm.PREC_FP64, 16,
                             merge=merge)
    for s in (one, many):
        s.advance(0, 2)
    _same(one, many, bx, N)
    b0, b1 = one.gw_spectrum(mode=1)[0], many.gw_spectrum(mode=1)[0]
    np.testing.assert_allclose(b0, b1, rtol=1e-12, atol=1e-15 * b0.max())


@MERGE
@pytest.mark.parametrize("interp", [1, 2, 4])
@pytest.mark.parametrize("integrator", [10, 21])
def test_finer_level_on_a_merged_base(integrator, interp, merge):
    """Ghost cells of level 1 from coarse cells of several boxes and through
    the periodic boundary, and its average-down onto them."""
    inp = complex_scalar(N=32, integrator=integrator, L=8.0, nghost=3,
                         **{"amr.max_refinement_levels": 1, "amr.te_crit": 1e-3,
                            "amr.regrid_dt": 0.05, "amr.interpolation_type": interp})
    lev1 = [[20, 20, 20, 43, 43, 43], [0, 2, 0, 9, 13, 11], [44, 20, 20, 55, 31, 31]]
    one, many, bx, N = _pair("ComplexScalar", inp, shm.PREC_FP64, 16, merge=merge)
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
