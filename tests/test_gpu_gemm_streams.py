"""Large products wherever they are called from - host threads that share a stream, many streams, graphs - give the bits of one
eager call: each has its workspace to itself from its first launch to its last."""
import ctypes as C
import threading

import numpy as np
import pytest

from tests.test_gpu_linear import lin, rocm  # noqa: F401  (fixtures)

pytestmark = pytest.mark.gpu

# by the plan: packed rows without slices of K, packed rows with slices of K, and a small product in slices on the fp32 tiles
SHAPES = [(48, 36000, 928), (128, 4096, 4096), (64, 128, 1600)]


@pytest.fixture(scope="module")
def hip():
    return C.CDLL("libamdhip64.so")


def ok(rc):
    assert rc == 0, f"HIP error {rc}"


class Product:
    """One product: its operands, a result buffer, and the bits an eager call gives."""

    def __init__(self, rocm, lin, shape, seed):  # noqa: F811
        self.M, self.N, self.K = shape
        rng = np.random.default_rng(seed)
        self.x = rocm.DeviceBuffer.from_numpy(rng.standard_normal((self.M, self.K), dtype=np.float32))
        w = rocm.DeviceBuffer.from_numpy(rng.standard_normal((self.N, self.K), dtype=np.float32))
        self.layer, self.out = lin.Linear(self.K, self.N, w, None), rocm.DeviceBuffer(self.M * self.N * 4)
        self.zero = np.zeros((self.M, self.N), np.float32)
        self.run(None)
        self.want = self.get()

    def run(self, stream):
        self.layer.Forward(self.x, (self.M, self.K), self.out, stream=stream)

    def get(self):
        return self.out.to_numpy(np.uint32, (self.M, self.N))

    def clear(self):
        from born_amd import _capi
        _capi.check(_capi.lib().born_rocm_h2d(self.out.ptr, self.zero.ctypes.data, self.zero.nbytes, None))

    def check(self, what):
        assert np.array_equal(self.get(), self.want), what
        self.clear()


@pytest.mark.parametrize("kind", ["null", "own", "per thread"])
def test_host_threads_on_one_stream(rocm, lin, hip, kind):  # noqa: F811
    stream = C.c_void_p({"null": None, "own": None, "per thread": 2}[kind])
    if kind == "own":
        ok(hip.hipStreamCreate(C.byref(stream)))
    products = [Product(rocm, lin, SHAPES[i % 3], i) for i in range(8)]
    for p in products:
        p.clear()
    start, wrong = threading.Barrier(8), []

    def work(p, i):
        start.wait()
        for _ in range(20):
            p.run(stream)
        ok(hip.hipStreamSynchronize(stream))               # (a thread's own stream, where there is one)
        if not np.array_equal(p.get(), p.want):
            wrong.append(i)

    threads = [threading.Thread(target=work, args=(p, i)) for i, p in enumerate(products)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    if kind == "own":
        ok(hip.hipStreamDestroy(stream))


def test_more_streams_than_keep_a_workspace(rocm, lin, hip):  # noqa: F811
    products = [Product(rocm, lin, s, 50 + i) for i, s in enumerate(SHAPES)]
    streams = [C.c_void_p() for _ in range(20)]
    for s in streams:
        ok(hip.hipStreamCreate(C.byref(s)))
    for s in streams:
        for p in products:
            p.clear()
            p.run(s)
        ok(hip.hipStreamSynchronize(s))
        for p in products:
            p.check(p.K)
    for s in streams:
        ok(hip.hipStreamDestroy(s))


def _capture(hip, stream, products):
    graph, gexec = C.c_void_p(), C.c_void_p()
    ok(hip.hipStreamBeginCapture(stream, 0))               # hipStreamCaptureModeGlobal
    for p in products:
        p.run(stream)
    ok(hip.hipStreamEndCapture(stream, C.byref(graph)))
    ok(hip.hipGraphInstantiate(C.byref(gexec), graph, None, None, C.c_size_t(0)))
    ok(hip.hipGraphDestroy(graph))
    return gexec


def test_graphs_replayed_beside_each_other_and_eager_products(rocm, lin, hip):  # noqa: F811
    """Two graphs captured on one stream that never ran a product before, replayed on two others while it runs eager ones."""
    sets = [[Product(rocm, lin, s, 100 + 10 * j + i) for i, s in enumerate(SHAPES)] for j in range(3)]
    s, s1, s2 = C.c_void_p(), C.c_void_p(), C.c_void_p()
    for x in (s, s1, s2):
        ok(hip.hipStreamCreateWithFlags(C.byref(x), 1))    # hipStreamNonBlocking: apart from the null stream
    g1, g2 = _capture(hip, s, sets[0]), _capture(hip, s, sets[1])
    for p in sets[0] + sets[1] + sets[2]:
        p.clear()
    for it in range(6):
        for _ in range(4):
            ok(hip.hipGraphLaunch(g1, s1))
            ok(hip.hipGraphLaunch(g2, s2))
            for p in sets[2]:
                p.run(s)
        ok(hip.hipDeviceSynchronize())
        for j in range(3):
            for p in sets[j]:
                p.check((it, j, p.K))
    for g in (g1, g2):
        ok(hip.hipGraphExecDestroy(g))
    # graph after graph: what they held comes back
    free, total, least = C.c_size_t(), C.c_size_t(), []
    for it in range(12):
        g = _capture(hip, s, sets[it % 3])
        ok(hip.hipGraphLaunch(g, s1))
        ok(hip.hipStreamSynchronize(s1))
        for p in sets[it % 3]:
            p.check((it, p.K))
        ok(hip.hipGraphExecDestroy(g))
        ok(hip.hipMemGetInfo(C.byref(free), C.byref(total)))
        least.append(free.value)
    assert least[2] - least[-1] < 200 << 20, least
    for x in (s, s1, s2):
        ok(hip.hipStreamDestroy(x))
