"""Host decisions of the products (born_amd/csrc/gemm_plan.cpp), without a GPU."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

WRAPPER = """
#include "gemm_plan.h"
extern "C" long long budget() { return born::GEMM_WS_MAX; }
// [tile, slices, kslice, rows, bytes]
extern "C" void plan(int M, int N, int K, long long *out) {
    const born::SplitPlan p = born::gemm_split_plan(M, N, K);
    out[0] = p.tile; out[1] = p.slices; out[2] = p.kslice; out[3] = p.rows;
    out[4] = p.rows ? born::gemm_split_bytes(p, p.rows < M ? p.rows : M, N, K) : 0;
}
extern "C" int pays(int M, int N, int K, long long ldb) { return born::gemm_split_pays(M, N, K, ldb); }
extern "C" int small(int M, int K, int N, int b_transposed, int whole, long long tiles) { return born::gemm_small_pays(M, N, K, b_transposed, whole, tiles); }
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "wrapper.cpp").write_text(WRAPPER)
    so, csrc = str(d / "libplan.so"), os.path.join(ROOT, "born_amd", "csrc")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-I", csrc, os.path.join(csrc, "gemm_plan.cpp"), str(d / "wrapper.cpp"), "-o", so])
    lib = C.CDLL(so)
    lib.budget.restype = C.c_longlong
    lib.pays.argtypes = [C.c_int, C.c_int, C.c_int, C.c_longlong]
    return lib


def test_pitches_beyond_32_bit_offsets_stay_on_the_fp32_tiles(plan):
    # the weights' loads: 16 + 4 (31 ldb + 31) bytes past a wave's first value, 16 bytes wide
    most = (2 ** 32 - 32 - 4 * 31) // (4 * 31)
    assert plan.pays(64, 32000, 4096, 4096) and plan.pays(64, 32000, 4096, 2 ** 25)
    for ldb in (most + 1, 35_000_000, 2 ** 32, 2 ** 40):
        assert not plan.pays(64, 35_000_000, 64, ldb), ldb
    for ldb in range(2 ** 25 - 2, 2 ** 25 + 3):
        assert not plan.pays(64, 32000, 4096, ldb) or ldb <= most, ldb


def _plan(plan, M, N, K):
    out = (C.c_longlong * 5)()
    plan.plan(M, N, K, out)
    return dict(zip(("tile", "slices", "kslice", "rows", "bytes"), out))


def test_plans_fit_the_workspace(plan):
    """What a plan asks for fits, and few products stay on the fp32 tiles for it: none that the rows of a hidden layer or a head make."""
    sizes = [33, 64, 65, 200, 256, 512, 708, 1024, 2048, 4096, 5000, 20001]
    seen = left = 0
    for M in sizes:
        for N in (1, 130, 1000, 2048, 4096, 8192, 10386, 14336, 32000, 128256, 152064):
            for K in (16, 61, 288, 1056, 2240, 3584, 4096, 8192, 14336, 65536, 160000):
                if not plan.pays(M, N, K, K):
                    continue
                p = _plan(plan, M, N, K)
                seen += 1
                if p["rows"] == 0:
                    left += K < 65536
                    assert K >= 65536 or N <= 1000, (M, N, K)
                    continue
                assert 0 < p["bytes"] <= plan.budget(), (M, N, K, p)
                assert p["rows"] == M or p["rows"] % (64, 128, 128, 256)[p["tile"]] == 0, (M, N, K, p)
                # slices of whole pairs of groups that cover K, none of them empty
                assert p["kslice"] % 64 == 0 and (p["slices"] - 1) * p["kslice"] < K <= p["slices"] * p["kslice"], (M, N, K, p)
    assert seen > 700 and left < 25
    for M, N, K in ((512, 4096, 4096), (1024, 4096, 4096), (2048, 4096, 4096), (256, 8192, 4096), (1024, 8192, 4096), (512, 14336, 4096),
                    (512, 4096, 14336), (256, 4096, 14336), (708, 10386, 2240)):
        assert _plan(plan, M, N, K)["rows"], (M, N, K)


def test_products_whose_rows_come_in_chunks(plan):
    """What tests/test_gpu_gemm_split.py multiplies in chunks of rows does come in chunks, with and without slices of K."""
    p = _plan(plan, 2900, 2600, 4096)
    assert p["slices"] == 1 and 1 < -(-2900 // p["rows"]) <= 3, p
    p = _plan(plan, 1900, 2600, 8192)
    assert 0 < p["rows"] < 1900, p
    p = _plan(plan, 700, 4096, 8192)
    assert p["slices"] > 1 and p["rows"] < 700, p
    assert _plan(plan, 64, 4096, 200000)["rows"] == 0


def test_sums_of_few_terms_stay_on_the_fp32_tiles(plan):
    assert plan.pays(4096, 65536, 16, 16) and not plan.pays(4096, 65536, 15, 15)


def test_a_long_k_of_few_squares_is_left_to_the_tiles_slices(plan):
    """A square has one CU, the tiles' slices of K have up to sixteen each: wherever that was measured the faster."""
    for M, K, N in ((16, 8193, 16), (64, 8193, 10), (40, 12001, 100), (200, 20001, 100), (757, 6001, 94), (64, 100003, 10)):
        assert not plan.small(M, K, N, 1, 0, 16), (M, K, N)
    for M, K, N in ((16, 40001, 16), (64, 20001, 64), (40, 12001, 100), (757, 6001, 94), (4, 100003, 700), (16, 1000001, 16)):
        assert not plan.small(M, K, N, 0, 0, 16), (M, K, N)
    for M, K, N in ((128, 4096, 256), (512, 8192, 64), (1100, 4096, 64), (16, 4096, 1000), (17, 1440, 2524), (18, 3808, 2301), (64, 2016, 1108), (17, 1056, 4696), (8, 1568, 11388)):   # K a multiple of 32
        assert not plan.small(M, K, N, 1, 1, 64) and not plan.small(M, K, N, 0, 1, 64), (M, K, N)
    for M, K, N in ((6, 4096, 2928), (14, 3616, 4000), (17, 960, 2594), (64, 1408, 1410), (128, 1472, 901), (200, 1280, 766), (6, 384, 8728), (64, 2048, 1024)):
        assert plan.small(M, K, N, 1, 1, 64) and plan.small(M, K, N, 0, 1, 64), (M, K, N)
    for M, K, N in ((16, 3211, 16), (64, 6001, 10), (40, 8193, 100), (200, 12001, 200), (400, 4097, 300), (911, 19590, 17), (3, 100003, 252)):
        assert plan.small(M, K, N, 1, 0, 16), (M, K, N)
    for M, K, N in ((16, 24001, 16), (64, 16001, 10), (40, 8193, 100), (256, 6001, 256), (3, 30001, 700)):
        assert plan.small(M, K, N, 0, 0, 16), (M, K, N)


def test_large_results_of_a_short_k_are_left_to_the_tiles(plan):
    for M, K, N in ((8000, 3, 8000), (4096, 7, 4000), (20000, 7, 2000)):
        assert not plan.small(M, K, N, 1, 0, 4000) and not plan.small(M, K, N, 0, 0, 4000), (M, K, N)
    assert not plan.small(4096, 20, 1000, 0, 0, 1024) and plan.small(4096, 20, 1000, 1, 0, 1024)
    assert plan.small(1000, 7, 4001, 1, 0, 1024) and plan.small(200000, 7, 33, 0, 0, 1563)                      # rows of odd length
