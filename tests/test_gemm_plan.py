"""Launch plans of the tiled GEMMs (csrc/q4_gemm_plan.hpp: host arithmetic, compiled here by itself)."""
import ctypes
import os
import subprocess

import pytest

from conftest import ROOT

WRAPPER = r"""
#include "q4_gemm_plan.hpp"
extern "C" void plan(int M, int red, int nout, size_t workspace, int* out) {
    const q4::GemmPlan p = q4::plan_gemm(M, red, nout, workspace);
    out[0] = p.cfg; out[1] = p.splits; out[2] = p.tail_cols; out[3] = p.tail_splits;
}
"""
NARROW128, NARROW, WIDE = 0, 2, 3            # 128 x 128, 256 x 128 and 256 x 256 tiles
ANY = 2 ** 62


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("plan")
    (tmp / "plan.cpp").write_text(WRAPPER)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I" + os.path.join(ROOT, "alpaca_lora_4bit_amd", "csrc"),
                           str(tmp / "plan.cpp"), "-o", str(tmp / "plan.so")])
    lib = ctypes.CDLL(str(tmp / "plan.so"))
    lib.plan.argtypes = [ctypes.c_int] * 3 + [ctypes.c_size_t, ctypes.POINTER(ctypes.c_int)]
    lib.plan.restype = None
    return lib


def _plan(lib, M, red, nout, workspace=ANY):
    out = (ctypes.c_int * 4)()
    lib.plan(M, red, nout, workspace, out)
    return tuple(out)


@pytest.mark.parametrize("M", [65, 100, 128])
@pytest.mark.parametrize("nout", [73728, 81920, 98304])
def test_up_to_128_rows_keep_the_128_row_tiles(plans, M, nout):
    """More wide tiles than CUs with a remainder, but half of every 256-row tile would be padding."""
    assert _plan(plans, M, 2048, nout)[0] == NARROW128
    assert _plan(plans, 129, 2048, nout)[0] == WIDE and _plan(plans, 129, 2048, nout)[2] > 0
