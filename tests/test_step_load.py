"""Lattices stepped at once: which of them may keep their step's data in the last-level cache (csrc/step_load.h),
and that the streamed and the cached passes of a single lattice give the same bits."""
import os
import subprocess
import threading

import numpy as np
import pytest

from axion_grav_amd import capi
from tests.conftest import ROOT, SQ_HALF, phys

PROGRAM = """
#include "step_load.h"
#include <thread>
#include <vector>
using namespace axg;
#define CHECK(c) do { if (!(c)) return __LINE__; } while (0)
static int64_t set(int64_t n, int comp) { return step_bytes(n * n * n, 8, comp ? 4 : 0, true); }
int main()
{
    CHECK(step_bytes(10, 16, 0, false) == 480 && step_bytes(10, 8, 4, true) == 1000);
    for (int comp = 0; comp < 2; comp++) {
        const StepLoad a(0, set(128, comp));
        CHECK(a.fits());
        {
            const StepLoad b(0, set(128, comp));
            CHECK(!a.fits() && !b.fits());
        }
        const StepLoad other(1, set(128, comp));  // another device
        CHECK(a.fits() && other.fits());
    }
    {
        const StepLoad a(0, set(96, 1)), b(0, set(96, 1));
        CHECK(a.fits() && b.fits());
        const StepLoad c(0, set(96, 1));
        CHECK(!a.fits() && !c.fits());
    }
    {
        const StepLoad a(0, set(512, 1)), b(0, set(96, 1));
        CHECK(!b.fits());
    }
    std::vector<std::thread> t;
    for (int i = 0; i < 8; i++)
        t.emplace_back([] { for (int k = 0; k < 100000; k++) StepLoad l(0, STEP_CACHE + k); });
    for (auto& x : t) x.join();
    const StepLoad last(0, STEP_CACHE);
    CHECK(last.fits());
    return 0;
}
"""


def test_lattices_share_the_cache(tmp_path):
    src, exe = tmp_path / "p.cpp", tmp_path / "p"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++20", "-O1", "-pthread", "-I", os.path.join(ROOT, "axion_grav_amd", "csrc"), str(src),
                    "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)], timeout=60).returncode == 0


def made(N, prec, seed, fix):
    L = capi.Lattice(capi.make_params(N, phys(N)["dspa"], SQ_HALF, precision=prec, gw_fix_swap=fix))
    L.init_flat(seed, 4.001 * phys(N)["dwav"])
    return L


def state(L):
    return (*L.get_fields(), *L.gw_state())


# the sizes whose passes have both forms; a batch's lattices that are no stack stream
@pytest.mark.gpu
@pytest.mark.parametrize("prec", [capi.FP32C, capi.FP32])
@pytest.mark.parametrize("N,fix", [(72, True), (96, False), (128, True)])
def test_streamed_matches_cached(N, fix, prec, monkeypatch):
    print("[case] streamed single lattice", N, fix, prec, flush=True)
    monkeypatch.setenv("AXG_BATCH_STACK", "0")
    with made(N, prec, 1, fix) as one, made(N, prec, 1, fix) as a:
        one.advance_steps(1.0, 0.05, 4)
        capi.batch_advance([a], 1.0, 0.05, 4, 2)
        for x, y in zip(state(one), state(a)):
            assert np.array_equal(x, y)


@pytest.mark.gpu
def test_two_threads_match_one():
    print("[case] two lattices stepped at once", flush=True)
    N, got = 128, {}

    def run(seed):
        with made(N, capi.FP32C, seed, False) as L:
            for k in range(3):
                L.advance_steps(1.0 + 0.5 * k, 0.01, 50)
            got.setdefault(seed, []).append(state(L))

    for s in (1, 2):
        run(s)
    t = [threading.Thread(target=run, args=(s,)) for s in (1, 2)]
    for x in t:
        x.start()
    for x in t:
        x.join()
    for one, both in got.values():
        for x, y in zip(one, both):
            assert np.array_equal(x, y)
