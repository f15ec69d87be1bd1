"""The workspace a handle takes when a call first wants it (born_amd/csrc/handle_workspace.h) against a stand-in for the HIP runtime, without a GPU:
a call under capture, memory that runs out, and the captures of other threads."""
import os
import subprocess

import pytest

from tests.test_gemm_workspace import HIP, ROOT

MAIN = r"""
#include "handle_workspace.h"
#include <cstdio>
#include <cstring>
using namespace born;
#define CHECK(x) do { if (!(x)) { std::printf("failed: %s (line %d)\n", #x, __LINE__); std::exit(1); } } while (0)
int main(int, char **argv) {
    hip_strict = true;                                 // every allocation in relaxed mode
    void *p = nullptr;
    bool refused = false;
    Stream s;
    if (!std::strcmp(argv[1], "capture")) {
        Graph g;
        s.capturing = &g;
        take_once(&s, 1000, &p, &refused);
        CHECK(!p && !refused && hip_mallocs == 0);
        s.capturing = nullptr;
        s.broken = true;                               // (a stream that cannot be asked)
        take_once(&s, 1000, &p, &refused);
        CHECK(!p && !refused && hip_mallocs == 0);
        s.broken = false;
        take_once(&s, 1000, &p, &refused);
        CHECK(p && !refused && hip_mallocs == 1);
        void *const first = p;
        take_once(&s, 1000, &p, &refused);
        CHECK(p == first && hip_mallocs == 1);
    } else if (!std::strcmp(argv[1], "no_memory")) {
        hip_full = true;
        take_once(&s, 1000, &p, &refused);
        CHECK(!p && refused && hip_live.empty());
        hip_full = false;
        take_once(&s, 1000, &p, &refused);             // not asked again
        CHECK(!p && hip_mallocs == 0);
    } else {
        take_once(nullptr, 1000, &p, &refused);
        CHECK(p && hip_mode == hipStreamCaptureModeGlobal);   // (the thread's mode is what it was)
    }
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("handle_workspace")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(HIP)
    (d / "main.cpp").write_text(MAIN)
    exe = str(d / "main")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-g", "-pthread", "-I", str(d), "-I", os.path.join(ROOT, "born_amd", "csrc"), str(d / "main.cpp"), "-o", exe])
    return exe


@pytest.mark.parametrize("what", ["capture", "no_memory", "null_stream"])
def test_handle_workspace(program, what):
    got = subprocess.run([program, what], capture_output=True, text=True, timeout=60)
    assert got.returncode == 0, got.stdout + got.stderr
