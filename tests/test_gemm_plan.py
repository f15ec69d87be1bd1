"""Host decisions of the large products (born_amd/csrc/gemm_plan.cpp), without a GPU."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

WRAPPER = """
#include "gemm_plan.h"
extern "C" int pays(int M, int N, int K, long long ldb) { return born::gemm_split_pays(M, N, K, ldb); }
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "wrapper.cpp").write_text(WRAPPER)
    so, csrc = str(d / "libplan.so"), os.path.join(ROOT, "born_amd", "csrc")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-I", csrc, os.path.join(csrc, "gemm_plan.cpp"), str(d / "wrapper.cpp"), "-o", so])
    lib = C.CDLL(so)
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
