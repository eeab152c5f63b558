"""The rule that picks the launch shape of untuned levels, on the CPU: every
set of built tile shapes (wide projects at radius 3 leave only the 32 x 8 tile,
or none, within the LDS budget) gets a shape the launches can take."""
import itertools
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NVAR, DEFAULT = 5, 1

MAIN = r"""
#include <cstdio>
#include "shm_launch_rule.hpp"
int main() {
    int integ, nf, R, f64, lo, gw, grp, ko, fuse, mask, fmask, fused, nbox;
    while (std::scanf("%d %d %d %d %d %d %d %d %d %d %d %d %d", &integ, &nf, &R, &f64, &lo, &gw,
                      &grp, &ko, &fuse, &mask, &fmask, &fused, &nbox) == 13) {
        std::vector<shm::Box3> boxes;
        for (int i = 0; i < nbox; ++i) {
            int n[3];
            if (std::scanf("%d %d %d", n, n + 1, n + 2) != 3) return 1;
            boxes.push_back({{0, 0, 0}, {n[0] - 1, n[1] - 1, n[2] - 1}});
        }
        shm::LaunchRule r{boxes, integ, nf, R, f64 != 0, lo != 0, gw != 0, grp != 0, ko != 0,
                          256, fuse != 0, {}, {}};
        for (int v = 0; v < shm::kNVar; ++v) {
            r.stage_built[v] = (mask >> v) & 1;
            r.fused_ty[v] = (fmask >> v) & 1 ? shm::kVariants[v].nw : 0;
        }
        const shm::LaunchCfg c = r.pick(fused);
        std::printf("%d %d %d %d\n", c.variant, c.tz, c.fused, c.fused_variant);
        std::fflush(stdout);
    }
    return 0;
}
"""


@pytest.fixture(scope="module")
def pick(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("rule")
    src, exe = d / "rule.cpp", d / "rule"
    src.write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-O1", "-fsanitize=undefined", "-fno-sanitize-recover",
                    "-I", os.path.join(ROOT, "sledgehamr_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)

    def run(cases):
        text = "".join(" ".join(str(int(v)) for v in c[:-1]) + f" {len(c[-1])} " +
                       " ".join(str(v) for b in c[-1] for v in b) + "\n" for c in cases)
        r = subprocess.run([str(exe)], input=text, capture_output=True, text=True)
        assert r.returncode == 0, r.stderr[-500:]
        out = [tuple(int(v) for v in line.split()) for line in r.stdout.splitlines()]
        assert len(out) == len(cases)
        return out
    return run


BOXES = [[(n, n, n)] for n in (1, 2, 5, 16, 33, 64, 100, 144, 260)] + \
        [[(17, 33, 9)], [(17, 33, 9), (64, 8, 70), (5, 65, 31)], [(16, 16, 16)] * 40]


def test_any_set_of_built_shapes(pick):
    cases = [(i, nf, R, p == 0, p == 3, 0, 0, 0, fuse, mask, 7 if fuse else 0, f, b)
             for i, nf, R, p, fuse, mask, f, b in itertools.product(
                 (10, 11, 21), (1, 2, 8), (1, 3), (0, 1, 3), (0, 1),
                 range(1 << NVAR), (-1, 0, 1), BOXES)]
    for c, (v, tz, fused, fv) in zip(cases, pick(cases)):
        mask, fuse, boxes = c[9], c[8], c[-1]
        assert 0 <= v < NVAR and 0 <= tz <= max(b[2] for b in boxes), c
        # A shape that is not built only as the default: the launch then takes
        # the nearest built one, or reports that none is.
        assert (mask >> v) & 1 or v == DEFAULT, c
        assert (fused, fv >= 0) in ((0, False), (1, True)) and (not fused or fuse), c


@pytest.mark.parametrize("mask", [0, 1 << 3])
def test_no_usable_shape_leaves_the_default(pick, mask):
    """Eight fields at radius 3 in FP64: nothing, or the 32 x 8 tile alone."""
    cases = [(10, 8, 3, 1, 0, 0, 0, 0, 0, mask, 0, -1, [(n, n, n)]) for n in (16, 64, 128)]
    assert all(r[:2] == (DEFAULT, 0) for r in pick(cases))


@pytest.mark.parametrize("integrator,prec", [(10, 3), (21, 3), (11, 3), (11, 0)])
def test_two_fields_in_fp64_keep_eight_rows(pick, integrator, prec):
    """112^3 to 128^3: chunks of 16 planes on 64 x 4 tiles, which load 2.1
    cells per cell at radius 2, took up to 1.15 times as long as the default."""
    def shape(n):
        return pick([(integrator, 2, 2, prec == 0, prec == 3, 0, 0, 0, 0, 31, 0, -1,
                      [(n, n, n)])])[0][:2]
    assert [shape(n) for n in (112, 120, 128)] == [(DEFAULT, 0)] * 3
    assert shape(48) == (0, 4) and shape(96) == (3, 8) and shape(136) == (3, 16)


@pytest.mark.parametrize("integrator", [10, 21])
def test_two_fields_in_fp64_keep_eight_rows_beside_the_fused_pass(pick, integrator):
    """The later stages of a fused FP64 step: 64 x 8 but for 4-plane chunks
    (176^3 on 64 x 4 tiles was slower than unfused)."""
    def shape(n):
        return pick([(integrator, 2, 2, 1, 0, 0, 0, 0, 1, 31, 7, -1, [(n, n, n)])])[0]
    for n in (80, 112, 142, 176, 256):
        assert shape(n)[0] == DEFAULT and shape(n)[2] == 1
    assert shape(64)[1] == 4 and shape(64)[0] != DEFAULT


def test_levels_just_short_of_filling_the_chip(pick):
    """130^3 to 136^3 are 255 tiles of 32 planes: chunks of 16 planes took up to
    1.27 times as long as automatic ones."""
    def shape(nf, R, integrator, prec, n):
        return pick([(integrator, nf, R, prec == 0, prec == 3, 0, 0, 0, 0, 31, 0, -1,
                      [(n, n, n)])])[0][:2]
    for n in (130, 132, 134):
        for prec in (1, 2, 3):
            for R in (1, 2, 3):
                assert shape(1, R, 21, prec, n) == (DEFAULT, 0)
                assert shape(1, R, 11, prec, n) == (DEFAULT, 0)
            assert shape(2, 2, 21, prec, n) == (DEFAULT, 0)
        assert shape(2, 2, 11, 0, n) == (3, 16)
    assert shape(1, 3, 21, 0, 136) == (DEFAULT, 0)
    assert shape(2, 2, 21, 2, 136) == (3, 16)
    # A corner of the chip stays to the model.
    assert shape(1, 2, 21, 2, 128)[1] == 8


def _gw(pick, integrator, prec, n):
    return pick([(integrator, 1, 3, prec == 0, prec == 3, 1, 1, 0, 0, 31, 0, -1,
                  [(n, n, n)])])[0][:2]


@pytest.mark.parametrize("integrator", [10, 21, 22])
@pytest.mark.parametrize("prec", [0, 1, 2, 3])
def test_gw_levels(pick, integrator, prec):
    """Chunks of 4 planes up to 64^3; at 110^3 to 120^3, where short chunks took
    up to 1.27 times as long, and above 256^3 the automatic ones."""
    for n in (32, 48, 64):
        assert _gw(pick, integrator, prec, n)[1] == 4
    for n in (110, 112, 120, 272, 384):
        v, z = _gw(pick, integrator, prec, n)
        assert v in (0, DEFAULT) and (z == 0 or z >= 14)
    for n in range(8, 258, 2):
        v, z = _gw(pick, integrator, prec, n)
        assert v in (0, DEFAULT, 3) and 0 <= z <= n


def _many(pick, nf, R, integrator, prec, boxes):
    return pick([(integrator, nf, R, prec == 0, prec == 3, 0, 0, 0, 0, 31, 0, -1, boxes)])[0][:2]


def test_many_boxes(pick):
    """Two fields in boxes 100 wide on 32-wide tiles took up to 1.45 times as
    long as on the default; boxes 32 wide do need them."""
    for prec in (1, 2, 3):
        assert _many(pick, 2, 2, 21, prec, [(100, 100, 100)] * 8) == (DEFAULT, 8)
        assert _many(pick, 2, 2, 21, prec, [(64, 70, 90)] * 7) == (DEFAULT, 0)
        assert _many(pick, 2, 2, 10, prec, [(32, 32, 32)] * 1000)[0] == 3
    assert _many(pick, 2, 2, 21, 0, [(90, 90, 90)] * 8) == (3, 8)
    assert _many(pick, 1, 2, 21, 2, [(128, 128, 128)] * 32) == (4, 16)
    assert _many(pick, 1, 1, 21, 2, [(64, 64, 64)] * 8) == (4, 4)
