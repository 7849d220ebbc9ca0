"""The launch rules (csrc/wrapper_plan.h, csrc/proj_plan.h), compiled for the host:
what the kernels read and write stays inside what the rules lay out, over the
sizes, stream counts, token counts and CU counts that the entry points take."""
import ctypes
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mhc_ascend_amd", "csrc")

SOURCE = r"""
#include "proj_plan.h"
#include "wrapper_plan.h"
extern "C" void stream_split(int64_t B, int64_t K, int np, int mt, int64_t slots, int64_t* out) {
    const mhc::StreamFill f = mhc::stream_fill_of(B, K, np, mt, 128, 64, slots);
    out[0] = mhc::stream_ksplit(f); out[1] = f.groups; out[2] = f.stages; out[3] = f.kmax;
    out[4] = mhc::stream_fill_splits(f);
}
extern "C" void bwd_split(int64_t B, int64_t C, int64_t dp_row, int64_t cus, int64_t* out) {
    out[0] = mhc::wbwd_split(B, C, dp_row, cus); out[1] = mhc::wbwd_tile(B, out[0]);
    out[2] = mhc::wbwd_max_tile(C, dp_row);
}
extern "C" void fold_split(int bf16, int64_t B, int64_t C, int np, int cus, int* out) {
    const mhc::WfoldSplit s = mhc::wfold_split(bf16, B, C, np, cus);
    out[0] = s.ks; out[1] = s.chunk; out[2] = s.steps;
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.cpp").write_text(SOURCE)
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror", "-shared", "-fPIC", f"-I{CSRC}",
                    str(d / "plan.cpp"), "-o", str(d / "plan.so")], check=True)
    return ctypes.CDLL(str(d / "plan.so"))


def _fold_split(plan, bf16, B, C, np, cus):
    out = (ctypes.c_int * 3)()
    plan.fold_split(int(bf16), ctypes.c_int64(B), ctypes.c_int64(C), np, cus, out)
    return tuple(out)


@pytest.mark.parametrize("cus", [1, 64, 256, 304])
@pytest.mark.parametrize("bf16", [False, True])
def test_fold_splits_all_hold_steps(plan, bf16, cus):
    """A split's prologue reads the packed Phi of its first step: it must be one
    of the packed steps.  All splits together cover every step, bf16 splits whole
    pairs of them."""
    for n in (2, 3, 4, 5, 6, 7, 8, 9, 12, 16, 17, 24, 32):
        for C in (8, 24, 40, 64, 72, 264, 1056, 1600, 2080, 4096, 4104, 7072, 7104, 7136, 7168, 8192, 16392, 1 << 21):
            for B in (1, 2, 16, 20, 63, 64, 65, 130, 511, 512, 1000, 2047, 2048, 5000, 65536):
                ks, chunk, steps = _fold_split(plan, bf16, B, C, n * n + 2 * n, cus)
                what = (n, C, B, ks, chunk, steps)
                assert ks >= 1 and chunk >= 1 and steps * 32 >= C, what
                assert (ks - 1) * chunk < steps <= ks * chunk, what
                assert not bf16 or chunk % 2 == 0, what


def test_stream_splits_are_those_of_the_full_search(plan):
    """The split count steps over counts that cannot win; trying every one in turn
    gives the same (rounds of workgroups x (stages per split + 3), a larger count
    only where that is 2% less)."""
    out = (ctypes.c_int64 * 5)()
    for n in (11, 12, 16, 24, 32, 48, 64):
        for C in (32, 64, 256, 512, 1280, 2048, 4096, 12288):
            for B in (1, 2, 7, 16, 32, 33, 64, 100, 128, 300, 512, 1000, 1500, 4096, 70000):
                for slots in (256, 512, 768):
                    mt = 4 if B > 32 else 2
                    plan.stream_split(ctypes.c_int64(B), ctypes.c_int64(n * C), n * n + 2 * n, mt,
                                      ctypes.c_int64(slots), out)
                    ks, groups, stages, kmax, fill = list(out)
                    assert groups == -(-B // (16 * mt)) * -(-(n * n + 2 * n) // 128) and stages == -(-n * C // 64)
                    assert kmax == max(1, min((stages + 1) // 2, -(-4096 // B))) and 1 <= fill <= kmax
                    best, best_cost = 1, None
                    for k in range(1, kmax + 1):
                        cost = -(-groups * k // slots) * (-(-stages // k) + 3)
                        if best_cost is None or cost * 50 < best_cost * 49:
                            best, best_cost = k, cost
                    assert ks == best, (n, C, B, slots, ks, best)


@pytest.mark.parametrize("cus", [1, 64, 256, 304])
def test_backward_tiles_all_hold_tokens(plan, cus):
    """Token tiles of the wrapper's backward: whole pipeline rounds that cover the
    tokens, none empty, and within the 2 GiB of a tile's buffers wherever that
    holds one round."""
    out = (ctypes.c_int64 * 3)()
    for n in (2, 5, 8, 12, 32):
        dp_row = -(-(n * n + 2 * n) // 32) * 32
        for C in (8, 64, 120, 1024, 1040, 4096, 7168, 16392, 100000, 1 << 20, 1_860_000, 1_900_032, 1 << 21):
            for B in (1, 31, 96, 97, 193, 1000, 2047, 4096, 24832, 65536, 1_000_003):
                plan.bwd_split(ctypes.c_int64(B), ctypes.c_int64(C), ctypes.c_int64(dp_row), ctypes.c_int64(cus), out)
                tiles, tile, most = list(out)
                what = (n, C, B, tiles, tile, most)
                assert tiles >= 1 and tile % 96 == 0 and (tiles - 1) * tile < B <= tiles * tile, what
                assert tile <= most or most < 96, what
