"""The kept device buffers (born_amd/csrc/device_pool.h) against a stand-in for the HIP runtime, without a GPU: the order they are given
back in, when all of them are, and allocations of the library where memory is short."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HIP = r"""
#pragma once
#include <cstdio>
#include <cstdlib>
#include <map>
#include <mutex>
#include <vector>
enum hipError_t { hipSuccess, hipErrorOutOfMemory, hipErrorInvalidValue, hipErrorUnknown };
inline std::mutex hip_mu;
inline std::map<void *, size_t> hip_live;
inline std::vector<void *> hip_freed;
inline size_t hip_capacity = (size_t)1 << 40, hip_used = 0;
inline int hip_refuse_frees = 0;
inline hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipMalloc(void **p, size_t n) {
    std::lock_guard<std::mutex> g(hip_mu);
    if (hip_used + n > hip_capacity) return hipErrorOutOfMemory;
    *p = std::malloc(1);
    hip_live[*p] = n;
    hip_used += n;
    return hipSuccess;
}
inline hipError_t hipFree(void *p) {
    std::lock_guard<std::mutex> g(hip_mu);
    if (hip_refuse_frees > 0) { hip_refuse_frees--; return hipErrorUnknown; }
    if (!hip_live.count(p)) return hipErrorInvalidValue;
    hip_used -= hip_live[p];
    hip_live.erase(p);
    hip_freed.push_back(p);
    return hipSuccess;                                    // (the memory stays ours: no address comes twice)
}
"""

MAIN = r"""
#include "device_pool.h"
#include <string>
#include <thread>
using namespace born;
#define CHECK(x) do { if (!(x)) { std::printf("failed: %s (line %d)\\n", #x, __LINE__); std::exit(1); } } while (0)
static void *get(DevicePool &p, size_t n) { void *x = nullptr; CHECK(p.alloc(n, &x) == hipSuccess && x); return x; }

// A buffer whose free the runtime refuses goes back to its place: the oldest is still the first to be given back.
static void order() {
    DevicePool p;
    void *hold = get(p, 1), *oldest = get(p, 4096), *small = get(p, 512), *more[300];
    CHECK(p.free(oldest) == hipSuccess && p.free(small) == hipSuccess);
    p.waited();
    hip_refuse_frees = 1;
    void *x = get(p, 4096);                               // asks for the smallest's free, is refused, gets a fresh one
    CHECK(x != oldest && hip_freed.empty());
    for (void *&m : more) m = get(p, 8192);
    for (void *m : more) CHECK(p.free(m) == hipSuccess);
    CHECK(hip_freed.size() >= 2 && hip_freed[0] == oldest && hip_freed[1] == small);
    CHECK(p.free(x) == hipSuccess && p.free(hold) == hipSuccess);
}
// The last buffer that comes back, of whatever size, takes all but 16 MiB of the kept ones with it, the oldest first.
static void last() {
    DevicePool p;
    void *large = get(p, (size_t)100 << 20), *tiny = get(p, 1), *a = get(p, 10 << 20), *b = get(p, 3000);
    CHECK(p.free(tiny) == hipSuccess && p.free(a) == hipSuccess && p.free(b) == hipSuccess && hip_live.size() == 4);
    p.waited();
    CHECK(get(p, 3000) == b && hip_freed.back() == tiny); // kept, and waited for: the smallest one's free
    CHECK(p.free(b) == hipSuccess && p.free(b) != hipSuccess);
    void *c = get(p, 12 << 20);
    CHECK(p.free(c) == hipSuccess && hip_live.size() == 4);
    CHECK(p.free(large) == hipSuccess && hip_live.size() == 2 && hip_freed.back() == a);
}
// Memory that is short: kept buffers make room for the library's own.
static void full() {
    void *hold, *x, *own = nullptr;
    DevicePool &p = device_pool();
    hip_capacity = 40 << 20;
    hold = get(p, 512);
    x = get(p, 30 << 20);
    CHECK(p.free(x) == hipSuccess && hip_used > (30u << 20));
    CHECK(device_malloc(&own, 20 << 20) == hipSuccess && hip_used < (21u << 20));
    CHECK(device_malloc(&own, 30 << 20) == hipErrorOutOfMemory);
    CHECK(p.free(hold) == hipSuccess);
}
static void threads() {
    DevicePool p;
    std::vector<std::thread> t;
    for (int k = 0; k < 8; k++)
        t.emplace_back([&] {
            for (int i = 0; i < 400; i++) {
                void *a = get(p, 512u << (i % 4)), *b = get(p, 700);
                CHECK(a != b && p.free(a) == hipSuccess && p.free(b) == hipSuccess);
                p.waited();
            }
        });
    for (auto &x : t) x.join();
    CHECK(hip_used <= (size_t)16 << 20);
}
int main(int, char **v) {
    const std::string t = v[1];
    if (t == "order") order();
    if (t == "last") last();
    if (t == "full") full();
    if (t == "threads") threads();
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("pool")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(HIP)
    (d / "main.cpp").write_text(MAIN)
    exe = str(d / "main")
    subprocess.check_call(["g++", "-O1", "-g", "-std=c++17", "-Wall", "-pthread", "-fsanitize=thread", "-I", str(d), "-I", os.path.join(ROOT, "born_amd", "csrc"),
                           str(d / "main.cpp"), "-o", exe])
    return exe


@pytest.mark.parametrize("what", ["order", "last", "full", "threads"])
def test_pool(program, what):
    got = subprocess.run([program, what], capture_output=True, text=True, timeout=120)
    assert got.returncode == 0, got.stdout + got.stderr
