"""The products' workspaces (born_amd/csrc/gemm_workspace.h) against a stand-in for the HIP runtime, without a GPU: threads that share a
stream, streams that come and go, captures and the graphs they leave, and memory that runs out."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HIP = r"""
#pragma once
#include <cstdlib>
#include <map>
#include <mutex>
#include <set>
#include <vector>
enum hipError_t { hipSuccess, hipErrorOutOfMemory, hipErrorInvalidValue, hipErrorUnknown };
enum hipStreamCaptureStatus { hipStreamCaptureStatusNone, hipStreamCaptureStatusActive, hipStreamCaptureStatusInvalidated };
enum hipStreamCaptureMode { hipStreamCaptureModeGlobal, hipStreamCaptureModeThreadLocal, hipStreamCaptureModeRelaxed };
enum { hipUserObjectNoDestructorSync = 1, hipGraphUserObjectMove = 1 };
struct Graph;
struct Object { void *x; void (*end)(void *); };
typedef Graph *hipGraph_t;
typedef Object *hipUserObject_t;
struct Stream { Graph *capturing = nullptr; unsigned long long id = 0; bool broken = false; };
typedef Stream *hipStream_t;
#define hipStreamPerThread ((hipStream_t)2)
struct Graph { std::vector<Object *> objects; };
inline std::mutex hip_mu;
inline std::set<void *> hip_live;
inline size_t hip_most = 0, hip_mallocs = 0;
inline bool hip_full = false;
inline thread_local hipStreamCaptureMode hip_mode = hipStreamCaptureModeGlobal;
inline bool hip_strict = false;                       // every allocation and free has to happen in relaxed mode
inline hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipMalloc(void **p, size_t) {
    std::lock_guard<std::mutex> g(hip_mu);
    if (hip_strict && hip_mode != hipStreamCaptureModeRelaxed) abort();
    if (hip_full) return hipErrorOutOfMemory;
    *p = std::malloc(1);
    hip_live.insert(*p);
    hip_mallocs++;
    if (hip_live.size() > hip_most) hip_most = hip_live.size();
    return hipSuccess;
}
inline hipError_t hipFree(void *p) {
    std::lock_guard<std::mutex> g(hip_mu);
    if (hip_strict && hip_mode != hipStreamCaptureModeRelaxed) abort();
    if (!hip_live.erase(p)) abort();
    std::free(p);
    return hipSuccess;
}
inline hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *m) { std::swap(*m, hip_mode); return hipSuccess; }
inline hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *st) {
    const bool real = s && s != hipStreamPerThread;
    if (real && s->broken) return hipErrorUnknown;
    *st = real && s->capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
inline hipError_t hipStreamGetCaptureInfo_v2(hipStream_t s, hipStreamCaptureStatus *st, unsigned long long *id, hipGraph_t *g, void *, void *) {
    *st = hipStreamCaptureStatusActive; *id = s->id; *g = s->capturing;
    return hipSuccess;
}
inline hipError_t hipUserObjectCreate(hipUserObject_t *o, void *x, void (*end)(void *), unsigned, unsigned) { *o = new Object{x, end}; return hipSuccess; }
inline hipError_t hipUserObjectRelease(hipUserObject_t o, unsigned) { o->end(o->x); delete o; return hipSuccess; }
inline hipError_t hipGraphRetainUserObject(hipGraph_t g, hipUserObject_t o, unsigned, unsigned) { g->objects.push_back(o); return hipSuccess; }
inline void graph_end(Graph *g) { for (Object *o : g->objects) { o->end(o->x); delete o; } delete g; }
"""

MAIN = r"""
#include "gemm_workspace.h"
#include <cstdio>
#include <cstring>
#include <string>
#include <thread>
using namespace born;
#define CHECK(x) do { if (!(x)) { std::printf("failed: %s (line %d)\n", #x, __LINE__); std::exit(1); } } while (0)
static void spin() { for (volatile int i = 0; i < 300; i++) {} std::this_thread::yield(); }

// Eight threads, one stream: a product writes its number to its workspace with its first launch and reads it with its last.
// The stream's order is the order of the calls here.
static void threads() {
    GemmWorkspaces w;
    Stream s;
    std::map<void *, int> memory;
    std::mutex m;
    std::vector<std::thread> t;
    bool bad = false;
    for (int k = 0; k < 8; k++)
        t.emplace_back([&, k] {
            for (int i = 0; i < 300; i++) {
                auto l = w.take(&s, 1000);
                if (!l.p) { bad = true; return; }
                { std::lock_guard<std::mutex> g(m); memory[l.p] = k; }
                spin();
                { std::lock_guard<std::mutex> g(m); if (memory[l.p] != k) bad = true; }
            }
        });
    for (auto &x : t) x.join();
    CHECK(!bad && hip_mallocs == 1);
}
// The per-thread stream: a buffer a thread, though the handle is one.
static void per_thread() {
    GemmWorkspaces w;
    void *a, *b;
    { auto l = w.take(hipStreamPerThread, 1); a = l.p; }
    std::thread([&] { auto l = w.take(hipStreamPerThread, 1); b = l.p; }).join();
    { auto l = w.take(hipStreamPerThread, 1); CHECK(l.p == a); }
    CHECK(a && b && a != b);
}
// More streams than are kept: all are served, the one unused longest gives way; a larger need replaces the buffer.
static void many_streams() {
    GemmWorkspaces w;
    Stream s[40];
    for (int r = 0; r < 3; r++)
        for (Stream &x : s) {
            { auto l = w.take(&x, 1); CHECK(l.p); }
            { auto l = w.take(&s[0], 1); CHECK(l.p); }
        }
    CHECK(hip_live.size() <= GemmWorkspaces::MAX_STREAMS && hip_most <= GemmWorkspaces::MAX_STREAMS + 1);
    size_t before = hip_mallocs;
    { auto l = w.take(&s[0], GEMM_WS_MIN + 1); CHECK(l.p); }
    { auto l = w.take(&s[0], GEMM_WS_MAX); CHECK(l.p); }
    { auto l = w.take(&s[0], 1); CHECK(l.p); }
    CHECK(hip_mallocs == before + 1 && hip_live.size() <= GemmWorkspaces::MAX_STREAMS);
    CHECK(!w.take(&s[0], GEMM_WS_MAX + 1).p);
}
// Captures: a buffer each, none of an eager stream's; given back once their graphs are gone.
static void captures() {
    GemmWorkspaces w;
    Stream s, other;
    void *eager, *first;
    { auto l = w.take(&s, 1); eager = l.p; }
    std::vector<Graph *> graphs;
    std::set<void *> seen{eager};
    for (unsigned long long id = 1; id <= 5; id++) {
        s.capturing = other.capturing = new Graph;
        s.id = other.id = id;
        { auto l = w.take(&s, 1); CHECK(l.p && seen.insert(l.p).second); first = l.p; }
        { auto l = w.take(&s, 100); CHECK(l.p == first); }                       // the next product of the capture
        { auto l = w.take(&other, 1); CHECK(l.p && seen.insert(l.p).second); }   // a branch on another stream
        { auto l = w.take(&s, GEMM_WS_MIN + 1); CHECK(l.p && seen.insert(l.p).second); }   // a larger one; the first stays the graph's
        graphs.push_back(s.capturing);
        s.capturing = other.capturing = nullptr;
    }
    { auto l = w.take(&s, 1); CHECK(l.p == eager); }
    CHECK(hip_live.size() == 16);
    for (Graph *g : graphs) graph_end(g);
    for (unsigned long long id = 6; id < 50; id++) {                             // graph after graph: no growth
        s.capturing = new Graph;
        s.id = id;
        { auto l = w.take(&s, 1); CHECK(l.p); }
        graph_end(s.capturing);
        s.capturing = nullptr;
        CHECK(hip_live.size() <= 2);
    }
}
static void no_memory() {
    GemmWorkspaces w;
    Stream s;
    hip_full = true;
    CHECK(!w.take(&s, 1).p);
    s.capturing = new Graph;
    CHECK(!w.take(&s, 1).p && s.capturing->objects.empty());
    s.capturing = nullptr;
    hip_full = false;
    CHECK(w.take(&s, 1).p);
    s.broken = true;
    CHECK(!w.take(&s, 1).p);
}
int main(int, char **v) {
    const std::string t = v[1];
    hip_strict = true;
    if (t == "threads") threads();
    if (t == "per_thread") per_thread();
    if (t == "many_streams") many_streams();
    if (t == "captures") captures();
    if (t == "no_memory") no_memory();
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("workspace")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(HIP)
    (d / "main.cpp").write_text(MAIN)
    exe = str(d / "main")
    subprocess.check_call(["g++", "-O1", "-g", "-std=c++17", "-Wall", "-pthread", "-fsanitize=thread", "-I", str(d), "-I", os.path.join(ROOT, "born_amd", "csrc"),
                           str(d / "main.cpp"), "-o", exe])
    return exe


@pytest.mark.parametrize("what", ["threads", "per_thread", "many_streams", "captures", "no_memory"])
def test_workspaces(program, what):
    got = subprocess.run([program, what], capture_output=True, text=True, timeout=120)
    assert got.returncode == 0, got.stdout + got.stderr
