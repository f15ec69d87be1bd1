"""Device buffers that are kept for the next of their size: contents, sizes at the edges of what is kept, a second free, and a
buffer that comes back while work on another stream still reads it."""
import ctypes as C
import threading

import numpy as np
import pytest

from born_amd import _capi

pytestmark = pytest.mark.gpu

MAX = 32 << 20                                             # the largest buffer that is kept


@pytest.fixture(scope="module")
def rocm():
    from born_amd import sampler as S
    assert S.DeviceCount() >= 1, "no HIP device visible"
    return S


@pytest.mark.parametrize("nbytes", [1, 511, 512, 513, MAX - 1, MAX, MAX + 1])
def test_live_buffers_are_apart(rocm, nbytes):
    for _ in range(3):
        a = [np.full(nbytes, i + 1, np.uint8) for i in range(4)]
        bufs = [rocm.DeviceBuffer.from_numpy(x) for x in a]
        for x, b in zip(a, bufs):
            assert np.array_equal(b.to_numpy(np.uint8, (nbytes,)), x)
        for b in bufs:
            b.free()


def test_more_buffers_than_are_kept(rocm):
    for _ in range(2):
        bufs = [rocm.DeviceBuffer.from_numpy(np.full(300, i, np.int32)) for i in range(300)]
        assert all((b.to_numpy(np.int32, (300,)) == i).all() for i, b in enumerate(bufs))
        for b in bufs:
            b.free()


def test_a_second_free_is_refused(rocm):
    p, lib = C.c_void_p(), _capi.lib()
    assert lib.born_rocm_alloc(4000, C.byref(p)) == 0
    assert lib.born_rocm_free(p) == 0
    assert lib.born_rocm_free(p) != 0


def test_freed_under_work_on_another_stream(rocm):
    """The other stream's copies of a buffer hold its contents, though the next buffer of its size is written at once."""
    hip, lib = C.CDLL("libamdhip64.so"), _capi.lib()
    n, copies = MAX // 4, 64                               # 64 copies take far longer than the host's next calls
    shape, side = np.array([n], np.int64), C.c_void_p()
    assert hip.hipStreamCreateWithFlags(C.byref(side), 1) == 0   # 1: hipStreamNonBlocking, apart from the null stream
    old, new = np.full(n, 1, np.float32), np.full(n, 2, np.float32)
    dst, other = [rocm.DeviceBuffer(4 * n) for _ in range(4)], rocm.DeviceBuffer.from_numpy(old[:16])
    for _ in range(3):
        src = rocm.DeviceBuffer.from_numpy(old)
        for i in range(copies):
            assert lib.born_rocm_reshape(src.ptr, shape.ctypes.data, 1, shape.ctypes.data, 1, dst[i % 4].ptr, side) == 0
        src.free()
        other.to_numpy(np.float32, (16,))                  # a wait, though not for the side stream
        nxt = rocm.DeviceBuffer.from_numpy(new)
        assert hip.hipStreamSynchronize(side) == 0
        for d in dst:
            assert (d.to_numpy(np.float32, (n,)) == 1).all()
        nxt.free()
    assert hip.hipStreamDestroy(side) == 0


def test_threads(rocm):
    bad = []

    def work(t):
        for i in range(200):
            x = np.full(64 * (1 + i % 5), 1000 * t + i, np.int32)
            b = rocm.DeviceBuffer.from_numpy(x)
            if not np.array_equal(b.to_numpy(np.int32, x.shape), x):
                bad.append((t, i))
            b.free()

    threads = [threading.Thread(target=work, args=(t,)) for t in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
