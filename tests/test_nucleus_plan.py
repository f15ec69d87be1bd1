"""Into how many parts rows without a top-k cut go (born_amd/csrc/nucleus_plan.h), without a GPU."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def parts(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "wrapper.cpp").write_text('#include "nucleus_plan.h"\nextern "C" int parts(int V, int rows, int most) { return born::row_parts(V, rows, most); }\n')
    so = str(d / "libplan.so")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-I", os.path.join(ROOT, "born_amd", "csrc"), str(d / "wrapper.cpp"), "-o", so])
    return C.CDLL(so).parts


@pytest.mark.parametrize("rows,V,n", [(3, 54166, 13), (32, 57142, 8), (42, 59999, 6), (51, 74999, 5), (64, 79999, 4), (85, 89999, 3), (128, 196608, 2)])
def test_the_shortest_rows_that_are_cut(parts, rows, V, n):
    assert parts(V, rows, 256) == n and parts(V - 1, rows, 256) == 0


def test_where_parts_were_measured_the_faster(parts):
    for rows, V in ((1, 57000), (1, 64001), (8, 61000), (32, 61000), (42, 66001), (64, 100003), (85, 100003), (1, 300000)):
        assert parts(V, rows, 256) >= 2, (rows, V)
    for rows, V in ((1, 50257), (32, 50257), (42, 57000), (64, 72000), (85, 80000), (128, 152064), (129, 300000)):
        assert parts(V, rows, 256) == 0, (rows, V)
    assert parts(300000, 4, 64) == 16 and parts(300000, 4, 7) == 0           # (a smaller workspace)
