"""The mean loss around the batch size from which its terms come in one copy: the per-row terms summed in fp32 in row order, bit for
bit, and what a target outside the classes does."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("classes", [10, 1000, 5000])
@pytest.mark.parametrize("batch", [1, 255, 256, 257, 3000])
def test_loss_is_the_terms_in_row_order(batch, classes):
    from born_amd import loss, sampler as S
    rng = np.random.default_rng(batch)
    x, t = (3 * rng.standard_normal((batch, classes))).astype(np.float32), rng.integers(0, classes, batch).astype(np.int32)
    x[0, (t[0] + 1) % classes] = np.inf
    d_x, d_t = S.DeviceBuffer.from_numpy(x), S.DeviceBuffer.from_numpy(t)
    s = S.NewSampler(S.SamplerConfig(), max_batch=batch, max_vocab=classes)
    total = np.float32(0)
    for v in S.token_logprobs_host(s, x, t):
        total = np.float32(total - v)
    ce = loss.CrossEntropyLoss(batch, classes)
    for _ in range(2):
        got = ce.Forward(d_x, (batch, classes), d_t)
        assert got.dtype == np.float32 and got.tobytes() == np.float32(total / np.float32(batch)).tobytes()
    bad = t.copy()
    bad[-1] = classes
    with pytest.raises(S.SamplerPanic, match="target index out of bounds"):
        ce.Forward(d_x, (batch, classes), S.DeviceBuffer.from_numpy(bad))
    assert ce.Forward(d_x, (batch, classes), d_t) == got     # (nothing is left of it)
    ce.Close()
    s.Close()


def _raw_loss(S, s, x, t, batch, classes, stream=None):
    import ctypes as C
    from born_amd import _capi
    out = C.c_float()
    _capi.check(_capi.lib().born_rocm_cross_entropy(s._h, x.ptr, batch, classes, t.ptr, C.byref(out), stream))
    return out.value


def test_loss_is_of_the_logits_as_they_are():
    """The handle's own settings are for its samples."""
    from born_amd import loss, sampler as S
    rng = np.random.default_rng(2)
    B, V = 5, 300
    x, t = S.DeviceBuffer.from_numpy(rng.standard_normal((B, V)).astype(np.float32)), S.DeviceBuffer.from_numpy(rng.integers(0, V, B).astype(np.int32))
    want = loss.CrossEntropyLoss(B, V).Forward(x, (B, V), t)
    s = S.NewSampler(S.SamplerConfig(Temperature=0.5, TopK=3, RepetitionPenalty=1.3, FrequencyPenalty=0.2), max_batch=B, max_vocab=V)
    assert np.float32(_raw_loss(S, s, x, t, B, V)).tobytes() == np.float32(want).tobytes()
    s.Close()


def test_loss_and_captures():
    """A stream under capture is refused before anything is recorded; a handle's first loss, which allocates, leaves another thread's capture alone."""
    import ctypes as C
    import threading

    from born_amd import _capi, sampler as S
    hip = C.CDLL("libamdhip64.so")
    rng = np.random.default_rng(3)
    B, V = 4, 64
    x, t = S.DeviceBuffer.from_numpy(rng.standard_normal((B, V)).astype(np.float32)), S.DeviceBuffer.from_numpy(rng.integers(0, V, B).astype(np.int32))
    tok, stream, other, graph, graph_exec = S.DeviceBuffer(4 * B), C.c_void_p(), C.c_void_p(), C.c_void_p(), C.c_void_p()
    assert hip.hipStreamCreate(C.byref(stream)) == 0 and hip.hipStreamCreateWithFlags(C.byref(other), 1) == 0
    s, fresh = (S.NewSampler(S.SamplerConfig(), max_batch=B, max_vocab=V) for _ in range(2))
    s.Argmax(x, B, V, tok, stream=stream)
    assert hip.hipStreamSynchronize(stream) == 0
    got = []
    assert hip.hipStreamBeginCapture(stream, 0) == 0          # 0: global, an unsafe call of any thread ends it
    try:
        with pytest.raises(_capi.BornRocmError) as e:
            _raw_loss(S, s, x, t, B, V, stream)
        th = threading.Thread(target=lambda: got.append(_raw_loss(S, fresh, x, t, B, V, other)))
        th.start()
        th.join()
        s.Argmax(x, B, V, tok, stream=stream)
    finally:
        rc = hip.hipStreamEndCapture(stream, C.byref(graph))
    assert e.value.code == _capi.ERR_UNSUPPORTED and "capture" in str(e.value)
    assert rc == 0 and graph.value, "the capture was invalidated"
    assert hip.hipGraphInstantiate(C.byref(graph_exec), graph, None, None, C.c_size_t(0)) == 0
    for _ in range(2):
        _capi.check(_capi.lib().born_rocm_h2d(tok.ptr, np.full(B, -1, np.int32).ctypes.data, 4 * B, None))
        assert hip.hipGraphLaunch(graph_exec, stream) == 0 and hip.hipStreamSynchronize(stream) == 0
        assert np.array_equal(tok.to_numpy(np.int32, (B,)), x.to_numpy(np.float32, (B, V)).argmax(1))
    assert got == [_raw_loss(S, s, x, t, B, V)]
    for f, h in ((hip.hipGraphExecDestroy, graph_exec), (hip.hipGraphDestroy, graph), (hip.hipStreamDestroy, stream), (hip.hipStreamDestroy, other)):
        f(h)
    s.Close()
    fresh.Close()
