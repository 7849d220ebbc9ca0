"""The wrapper's launch rules (csrc/wrapper_plan.h), compiled for the host: what
the kernels read and write stays inside what the rules lay out, over the sizes,
stream counts, token counts and CU counts that the entry points take."""
import ctypes
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mhc_ascend_amd", "csrc")

SOURCE = r"""
#include "wrapper_plan.h"
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
