"""The stage records of a step travel in one copy: more eager steps than the
record ring holds groups, and replayed steps, give the same cells with
parameters that change every stage (the 2/eta damping), for every integrator
of the project and on a level with coarse/fine ghost cells."""
import numpy as np
import pytest

import sledgehamr_amd as shm
from cases import complex_scalar

pytestmark = pytest.mark.gpu


def _run(integrator, graphs, steps, sync_every=0, lev1=None):
    extra = {"amr.max_refinement_levels": 1} if lev1 else {}
    sim = shm.Simulation("ComplexScalar", complex_scalar(N=16, integrator=integrator, **extra),
                         precision=shm.PREC_FP64)
    if lev1:
        sim.set_boxes(1, lev1)
        sim.init_state(1, 1, 4, [0.05])
    sim.init_state(0, 1, 3, [0.05])
    sim.set_graphs(graphs)
    for s in range(steps):
        if lev1:
            sim.evolve(1)
        else:
            sim.advance(0, 1)
        if sync_every and s % sync_every == 0:
            sim.sync()
    return [sim.download(lev, c) for lev in range(2 if lev1 else 1) for c in range(4)]


@pytest.mark.parametrize("integrator", [10, 11, 21, 22])
def test_many_steps(integrator):
    ref = _run(integrator, False, 300, sync_every=1)
    for graphs in (False, True):
        for a, b in zip(ref, _run(integrator, graphs, 300)):
            assert np.isfinite(a).all() and np.array_equal(a, b)


@pytest.mark.parametrize("integrator", [10, 21])
def test_fine_level(integrator):
    box = [[8, 8, 8, 23, 23, 23]]
    ref = _run(integrator, False, 40, sync_every=1, lev1=box)
    for graphs in (False, True):
        for a, b in zip(ref, _run(integrator, graphs, 40, lev1=box)):
            assert np.isfinite(a).all() and np.array_equal(a, b)
