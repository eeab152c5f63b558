"""Transfers through rings of slots, on the CPU with slots that a host thread
fills: every byte arrives whatever the size and however many threads can be
started, and the copying threads take no processor time while the device still
works on what was queued before.  The pool frees its rings with its last user,
also after one whose construction failed."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MIB = 1 << 20

MAIN = r"""
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <ctime>
#include <system_error>
#include "shm_to_host.hpp"
using namespace shm;

static unsigned char value(size_t i) { return (unsigned char)(i * 2654435761u >> 13); }

// bytes, milliseconds the first slot takes, threads that can be started
static int transfer(int, char **v) {
    const size_t n = std::strtoull(v[2], nullptr, 10);
    const int ms = std::atoi(v[3]);
    int threads = std::atoi(v[4]);
    std::vector<char> out(n + 1, 0), slots(kIoSlot * kIoSlots);
    const std::clock_t c0 = std::clock();
    std::clock_t fill = 0;  // the producer's own time
    copy_through_slots(out.data(), n, slots.data(),
        [&](size_t o, size_t b, int s) {
            const std::clock_t f0 = std::clock();
            for (size_t i = 0; i < b; ++i) slots[s * kIoSlot + i] = (char)value(o + i);
            fill += std::clock() - f0;
        },
        [&](int) {
            static bool first = true;
            if (first) std::this_thread::sleep_for(std::chrono::milliseconds(ms));
            first = false;
        },
        [&](auto f) {
            if (threads-- <= 0)
                throw std::system_error(
                    std::make_error_code(std::errc::resource_unavailable_try_again));
            return std::thread(f);
        });
    const std::clock_t used = std::clock() - c0 - (ms ? fill : 0);
    for (size_t i = 0; i < n; ++i)
        if ((unsigned char)out[i] != value(i)) return std::printf("byte %zu\n", i), 1;
    if (out[n]) return std::printf("past the end\n"), 1;
    std::printf("%.3f\n", (double)used / CLOCKS_PER_SEC);
    return 0;
}

struct Ring {
    size_t bytes;
    int device;
    int *freed;
    void reset() { ++*freed; }
};

struct Context {
    PoolUser<IoPool<Ring>> user;
    Context(IoPool<Ring> &p, bool fail) : user(p) {
        if (fail) throw 1;
    }
};

static int pool() {
    IoPool<Ring> p;
    int made = 0, freed = 0;
    auto make = [&](size_t b, int d) { return ++made, Ring{b, d, &freed}; };
    try {
        Context c(p, true);
    } catch (int) {
    }
    {
        Context a(p, false);
        {
            Context b(p, false);
            p.give(p.take(5, 0, make));
            p.give(p.take(5, 0, make));      // the kept one
            p.give(p.take(5, 1, make));      // another device
        }
        std::printf("%d %d ", made, freed);  // a user is left: kept
    }
    std::printf("%d %d ", made, freed);
    p.give(p.take(5, 0, make));              // no user: not kept
    std::printf("%d %d\n", made, freed);
    return 0;
}

int main(int argc, char **argv) {
    return argc == 2 ? pool() : transfer(argc, argv);
}
"""


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("to_host")
    src, out = d / "t.cpp", d / "t"
    src.write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-O2", "-pthread", "-I",
                    os.path.join(ROOT, "sledgehamr_amd", "csrc"), str(src), "-o", str(out)],
                   check=True)

    def run(*args):
        r = subprocess.run([str(out), *map(str, args)], capture_output=True, text=True,
                           timeout=120)
        assert r.returncode == 0, r.stdout + r.stderr
        return r.stdout.split()
    return run


@pytest.mark.parametrize("n", [2 * MIB + 1, 8 * MIB - 1, 8 * MIB, 8 * MIB + 1, 32 * MIB,
                               32 * MIB + 5, 75 * MIB + 3])
@pytest.mark.parametrize("threads", [8, 2, 1, 0])
def test_every_byte_arrives(exe, n, threads):
    exe("transfer", n, 0, threads)


def test_threads_do_not_spin_before_the_first_slot(exe):
    """0.6 s until the first slot is there.  Copying 30 MiB takes some 10 ms of
    processor time; one thread that polls would use 0.6 s."""
    assert float(exe("transfer", 30 * MIB, 600, 8)[0]) < 0.3


def test_pool_frees_its_rings_with_its_last_user(exe):
    assert exe("pool") == ["2", "0", "2", "2", "3", "3"]
