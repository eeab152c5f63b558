"""Transfers to the host through the pinned ring: exact values at the edges of
its units (2 MiB), slots (8 MiB) and of the ring itself (32 MiB), from several
threads at once, and the tag mask against the allocation-free path."""
import threading

import numpy as np
import pytest

import sledgehamr_amd as shm
from cases import complex_scalar, real_scalar

pytestmark = pytest.mark.gpu

ANY = {"shm.allow_any_grid_size": 1}


def _round_trip(N, seed):
    sim = shm.Simulation("RealScalar", real_scalar(N=N, **ANY), precision=shm.PREC_FP64)
    d = np.random.default_rng(seed).standard_normal(N ** 3)
    sim.upload(0, 1, d)
    ok = np.array_equal(sim.download(0, 1), d) and not sim.download(0, 0).any()
    sim.close()
    return ok


# 64^3 doubles are one unit; 102^3 pass one slot, 164^3 the ring.
@pytest.mark.parametrize("N", [2, 62, 64, 66, 102, 164])
def test_download_equals_upload(N):
    assert _round_trip(N, N)


def test_downloads_from_several_threads():
    res = {}

    def work(i):
        res[i] = all(_round_trip(n, 10 * i + n) for n in (64, 130, 66, 164))
    thr = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    for t in thr:
        t.start()
    for t in thr:
        t.join()
    assert res == {0: True, 1: True, 2: True}


@pytest.mark.parametrize("N", [32, 164])
def test_tag_mask_equals_direct_copy(N):
    inp = complex_scalar(N=N, **{**ANY, "amr.te_crit": 1e-3, "project.tag_strings": 1})
    sim = shm.Simulation("ComplexScalar", inp, precision=shm.PREC_FP32C16)
    sim.init_state(0, 1, 3, [0.05])
    sim.advance(0, 1)
    sim.create_shadow()
    sim.advance(0, 1)
    m0, c0, te = sim.te_tag(0, shm.TE_COMPUTE | shm.TE_TAGS, want_te=True)
    m1, c1 = sim.te_tag_noalloc(0)
    assert m0.any() and np.array_equal(m0, m1) and np.array_equal(c0, c1)
    assert te.shape == (4, N ** 3 // 8) and np.isfinite(te).all()
    assert int((te >= 1e-3).sum()) * 8 == int(c0[2:].sum())
