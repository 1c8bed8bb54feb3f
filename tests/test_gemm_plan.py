"""Launch plans of the tiled GEMMs (csrc/q4_gemm_plan.hpp: host arithmetic, compiled here by itself)."""
import ctypes
import os
import subprocess

import pytest

from conftest import ROOT

WRAPPER = r"""
#include "q4_gemm_plan.hpp"
extern "C" void plan(int M, int red, int nout, size_t workspace, int indexed, int* out) {
    const q4::GemmPlan p = q4::plan_gemm(M, red, nout, workspace, indexed == 1, indexed == 2);       // 2: forward, sequential groups
    out[0] = p.cfg; out[1] = p.splits; out[2] = p.tail_cols; out[3] = p.tail_splits;
}
extern "C" void group_plan(int fwd, int n, int M, int K, const int* N, int* out) {
    const q4::GroupPlan p = q4::plan_gemm_group(fwd, n, M, K, N);
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
    lib.plan.argtypes = [ctypes.c_int] * 3 + [ctypes.c_size_t, ctypes.c_int, ctypes.POINTER(ctypes.c_int)]
    lib.group_plan.argtypes = [ctypes.c_int] * 4 + [ctypes.POINTER(ctypes.c_int)] * 2
    lib.plan.restype = lib.group_plan.restype = None
    return lib


def _plan(lib, M, red, nout, workspace=ANY, indexed=False):
    out = (ctypes.c_int * 4)()
    lib.plan(M, red, nout, workspace, int(indexed), out)
    return tuple(out)


def _group_plan(lib, fwd, M, K, Ns):
    out = (ctypes.c_int * 4)()
    lib.group_plan(fwd, len(Ns), M, K, (ctypes.c_int * len(Ns))(*Ns), out)
    return tuple(out)


@pytest.mark.parametrize("M", [65, 100, 128])
@pytest.mark.parametrize("nout", [73728, 81920, 98304])
def test_up_to_128_rows_keep_the_128_row_tiles(plans, M, nout):
    """More wide tiles than CUs with a remainder, but half of every 256-row tile would be padding."""
    assert _plan(plans, M, 2048, nout)[0] == NARROW128
    assert _plan(plans, 129, 2048, nout)[0] == WIDE and _plan(plans, 129, 2048, nout)[2] > 0


def _partials(plan, M, nout):
    cfg, splits, tail_cols, tail_splits = plan
    if tail_cols:
        return 4 * tail_splits * M * tail_cols * 128 if tail_splits > 1 else 0
    return 4 * splits * M * nout if splits > 1 else 0


@pytest.mark.parametrize("M,red,nout", [(1969, 4352, 9472), (1576, 9600, 12800), (2605, 4352, 8704), (3950, 6784, 12800), (2048, 4096, 11008)])
def test_indexed_groups_have_no_wide_remainder_route(plans, M, red, nout):
    assert _plan(plans, M, red, nout)[0] == WIDE and _plan(plans, M, red, nout)[2] > 0
    assert _plan(plans, M, red, nout, indexed=True)[0] == NARROW


def test_a_plan_stays_inside_its_output_and_its_workspace(plans):
    """Every plan over rows, features and scratch sizes: the second launch's columns lie inside the output, no share is
    without a step, the partial sums fit the scratch given, and the query's size holds the plan of either group order."""
    import random
    from alpaca_lora_4bit_amd import _lib
    rng = random.Random(3)
    L = _lib.lib()
    for _ in range(4000):
        M = int(2 ** rng.uniform(0, 14))
        red, nout = 128 * int(2 ** rng.uniform(0, 7.5)), 128 * int(2 ** rng.uniform(0, 10))
        for indexed in (False, True, 2):
            whole = _plan(plans, M, red, nout, indexed=indexed)
            if indexed == 2 and nout % 256 == 0 and whole[0] == NARROW and whole[2] % 2:
                assert whole[3] * whole[2] // (whole[2] + 1) < 2
            assert _partials(whole, M, nout) <= L.q4_gemm_workspace_bytes(1, M, red, nout)
            scratch = rng.choice([0, 1 << 20, _partials(whole, M, nout), max(_partials(whole, M, nout) - 1, 0)])
            for p, room in ((whole, ANY), (_plan(plans, M, red, nout, scratch, indexed), scratch)):
                cfg, splits, tail_cols, tail_splits = p
                width = 256 if cfg == WIDE else 128
                assert nout % width == 0 and 0 <= tail_cols * 128 < nout and (nout - tail_cols * 128) % width == 0
                assert 1 <= splits <= max(red // 64, 1) and 1 <= tail_splits <= red // 64
                assert splits == 1 or tail_cols == 0
                assert _partials(p, M, nout) <= room


@pytest.mark.parametrize("M,red,nout,odd,even", [(1536, 4096, 11008, (1, 8), (2, 4)), (3328, 13824, 5120, (1, 8), (2, 4)),
                                                 (520, 1024, 11008, (1, 2), (1, 2)), (1024, 1024, 11136, (23, 2), (23, 2))])
def test_forward_remainders_are_planned_as_they_are_launched(plans, M, red, nout, odd, even):
    """Whole pairs of column tiles where the output has them and two shares are left; an odd width and one share keep the odd remainder."""
    assert _plan(plans, M, red, nout) == (NARROW, 1, *odd) == _plan(plans, M, red, nout, indexed=True)
    assert _plan(plans, M, red, nout, indexed=2) == (NARROW, 1, *even)


@pytest.mark.parametrize("M,K,Ns,was", [
    (1006, 8832, (9600, 9600, 9600), (NARROW, 1, 0, 1)),             # 276 narrow tiles: 1.08 rounds
    (846, 10368, (11392, 11392, 11392), (NARROW, 1, 0, 1)),          # 324
    (1086, 8064, (3712, 3712, 3712, 3712), (NARROW, 1, 0, 1)),       # 315
])
def test_grouped_grad_input_does_not_leave_a_second_round_nearly_empty(plans, M, K, Ns, was):
    """Widths without wide tiles just beyond one round of narrow ones: a remainder launch (1.23..1.28 times faster)."""
    cfg, splits, tail_cols, tail_splits = _group_plan(plans, 0, M, K, Ns)
    row_tiles = (M + 255) // 256
    assert (cfg, splits, tail_cols, tail_splits) != was
    assert tail_cols > 0 and tail_splits > 1 and (K // 128 - tail_cols) * row_tiles <= 256


def test_a_grouped_plan_stays_inside_its_output_and_its_workspace(plans):
    import random
    from alpaca_lora_4bit_amd import _lib
    rng = random.Random(4)
    L = _lib.lib()
    seen = set()
    for _ in range(6000):
        n = rng.choice([2, 3, 4])
        M, K = int(2 ** rng.uniform(7, 15)), 128 * int(2 ** rng.uniform(0, 8))
        Ns = [128 * int(2 ** rng.uniform(0, 8)) for _ in range(n)]
        arr = (ctypes.c_int * n)(*Ns)
        for fwd in (0, 1):
            cfg, splits, tail_cols, tail_splits = p = _group_plan(plans, fwd, M, K, Ns)
            assert bool(L.q4_gemm_grouped_applicable(fwd, n, M, K, arr)) == (cfg >= 0)
            if cfg < 0:
                assert M <= 128 or fwd
                continue
            seen.add((fwd, cfg, splits > 1, tail_cols > 0, tail_splits > 1))
            columns, steps = (sum(Ns), K // 64) if fwd else (K, sum(Ns) // 64)
            width = 256 if cfg == WIDE else 128
            assert all(c % width == 0 for c in (Ns if fwd else [K]))
            assert 0 <= tail_cols * 128 < columns and (columns - tail_cols * 128) % width == 0
            assert 1 <= splits <= 8 and 1 <= tail_splits <= 8 and max(splits, tail_splits) <= steps
            assert (splits == 1 or tail_cols == 0) and (tail_splits == 1 or tail_cols > 0)
            want = _partials(p, M, columns)
            assert L.q4_gemm_grouped_workspace_bytes(fwd, n, M, K, arr) == want and (want == 0 or not fwd)
    # what the estimate can choose came up: both widths, whole and split, and a remainder launch, split or not
    whole, split, rest, rest_split = (False, False, False), (True, False, False), (False, True, False), (False, True, True)
    assert {(0, NARROW, *k) for k in (whole, split, rest_split)} | {(0, WIDE, *k) for k in (whole, split, rest, rest_split)} <= seen
