"""How causal attention's query tiles are cut into runs (csrc/flash_plan.h): host code, compiled here alone and asked for a card of 256 CUs."""

from __future__ import annotations

import ctypes as C
import os
import subprocess

import pytest

from tests import flash_cuts

CSRC = os.path.join(os.path.dirname(__file__), "..", "pygpukit_amd", "csrc")
SHIM = """
#include "flash_plan.h"
using namespace pgk;
extern "C" void cut(int hq, int q_len, int kv_len, int d, int granted, int* out) {
    const FlashPlan even = flash_even_plan(256, (long long)fl_ceil_div(q_len, FL_BQ) * hq, q_len, kv_len, 16);
    int asked = 0;
    const FlashPlan p = flash_granted(flash_plan(256, even, hq, q_len, kv_len, d, 16), even, [&](int runs) { ++asked; return runs <= granted; });
    const int v[] = {p.runs, p.run, p.sides, even.runs, asked};
    for (int i = 0; i < 5; ++i) out[i] = v[i];
}
"""


@pytest.fixture(scope="module")
def cut(tmp_path_factory):
    at = tmp_path_factory.mktemp("flash_plan")
    (at / "shim.cpp").write_text(SHIM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-shared", "-fPIC", "-I", CSRC, "-o", str(at / "shim.so"), str(at / "shim.cpp")], check=True)
    lib = C.CDLL(str(at / "shim.so"))

    def ask(hq, q_len, kv_len, d=128, granted=16):
        out = (C.c_int * 5)()
        lib.cut(hq, q_len, kv_len, d, granted, out)
        return dict(zip(("runs", "run", "sides", "even", "asked"), out))

    return ask


@pytest.mark.parametrize("hq,n,tiles_of_a_run,runs,even", [(16, 1404, 10, 3, 2), (7, 1404, 4, 6, 4), (4, 1600, 4, 7, 6), (1, 3957, 4, 16, 8)])
def test_refused_scratch_leaves_the_even_cut_that_takes_less(cut, hq, n, tiles_of_a_run, runs, even):
    """A pool that refuses the rows of the heaviest tile's runs, but holds as many as the even cut has, gets that one; only below it one run."""
    for granted in range(1, 17):
        got = cut(hq, n, n, granted=granted)
        want = (runs, tiles_of_a_run) if granted >= runs else (even, 0) if granted >= even else (1, 0)
        assert (got["runs"], got["run"], got["even"]) == (*want, even), (granted, got)
        assert got["sides"] == 1 and got["asked"] <= 2


def test_calls_of_one_run_ask_for_no_scratch(cut):
    for hq, q_len, kv_len in ((26, 1250, 1250), (32, 1531, 1531), (32, 4096, 4096), (16, 400, 400), (64, 900, 900)):
        got = cut(hq, q_len, kv_len, granted=1)
        assert (got["runs"], got["run"], got["asked"]) == (1, 0, 0), got


@pytest.mark.parametrize("hq,q_len,kv_len,d,even,run", [(1, 1200, 1200, 128, 6, 0), (1, 1531, 1531, 128, 8, 0), (2, 1000, 1240, 128, 6, 0), (1, 1700, 1700, 128, 8, 0), (1, 1800, 1800, 128, 8, 4), (2, 1200, 1200, 128, 6, 4),
                                                        (1, 1250, 1250, 64, 7, 0), (1, 3000, 3000, 64, 8, 0), (1, 3100, 3100, 64, 8, 4), (2, 1400, 1400, 64, 7, 0), (4, 1400, 1400, 64, 6, 4)])
def test_few_workgroups_keep_the_even_cut(cut, hq, q_len, kv_len, d, even, run):
    """Both sides of the line for each head dim: even runs that occupy 7/16 (head dim 64: 3/4) of the CUs or fewer stay."""
    got = cut(hq, q_len, kv_len, d)
    assert (got["even"], got["run"]) == (even, run), got
    assert (16 * even * -(-q_len // 128) * hq <= (12 if d == 64 else 7) * 256) == (run == 0)


@pytest.mark.parametrize("cuts", ["SIDES", "ANY_COUNT", "MERGES", "FEW_WORKGROUPS", "EQUAL_TILES"])
def test_shapes_the_kernels_are_tested_with_are_cut_as_listed(cut, cuts):
    """Each of the GPU tests' shapes takes the route that it stands for."""
    for (hq, _, q_len, kv_len, d), want in getattr(flash_cuts, cuts).items():
        got = cut(hq, q_len, kv_len, d)
        assert (got["runs"], got["run"], got["sides"]) == want, (hq, q_len, kv_len, d, got)
