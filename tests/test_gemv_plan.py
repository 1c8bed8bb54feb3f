"""Split of the weight-streaming product (csrc/q4_gemv_plan.hpp: host arithmetic, compiled here by itself)."""
import ctypes
import os
import subprocess

import pytest

from conftest import ROOT

WRAPPER = r"""
#include "q4_gemv_plan.hpp"
extern "C" int blocks_per_workgroup(int M, int blocks, int strips, int groupsize) {
    return q4::plan_stream_blocks(M, blocks, strips, groupsize);
}
extern "C" int stream_takes(int M, int blocks, int strips, int groupsize) { return q4::plan_stream_takes(M, blocks, strips, groupsize); }
extern "C" long slab(int M, int nb) { return (long)q4::stream_slab_bytes(M, nb); }
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("plan")
    (tmp / "plan.cpp").write_text(WRAPPER)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I" + os.path.join(ROOT, "alpaca_lora_4bit_amd", "csrc"),
                           str(tmp / "plan.cpp"), "-o", str(tmp / "plan.so")])
    lib = ctypes.CDLL(str(tmp / "plan.so"))
    lib.slab.restype = ctypes.c_long
    return lib


@pytest.mark.parametrize("groupsize", [32, 64, 128, 4096])
def test_every_split_fits_the_arrival_count_and_the_lds(plan, groupsize):
    for M in range(1, 17):
        for blocks in list(range(1, 40)) + [254, 255, 256, 257, 510, 511, 1020]:
            for strips in (1, 2, 15, 16, 32, 64, 80, 128, 172, 192, 216, 240, 256, 257, 344, 512, 2000):
                nb = plan.blocks_per_workgroup(M, blocks, strips, groupsize)
                splits = -(-blocks // nb)
                assert 1 <= nb <= blocks and splits <= 255
                # beside the activation tiles (32 KB) within the 160 KB of a compute unit
                assert nb == 1 or plan.slab(M, nb) <= 128 * 1024
                assert nb == 1 or blocks > 255 or (strips * splits <= 256 and groupsize % 128 == 0 and M >= 5)
                # the fixed-point exchange below the arrival count: a workgroup adds up to twice its bias
                if plan.stream_takes(M, blocks, strips, groupsize):
                    assert splits * 2 * (nb << 46 if nb > 1 and splits * nb <= 511 else 1 << 47) < 2 ** 56
                else:
                    assert blocks * 2 ** 48 < 2 ** 56
