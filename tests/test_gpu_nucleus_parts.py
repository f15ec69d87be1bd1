"""Rows without a top-k cut that several workgroups share: lengths around the smallest that is cut and with ragged last parts, batches
from one row to the last that is cut in two, histories whose ids fall into every part, and the rows that are handed to one workgroup.
Against the oracle's fixed-point layer, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rocm():
    from born_amd import sampler as S
    assert S.DeviceCount() >= 1, "no HIP device visible"
    return S


def _check(oracle, rocm, x, u, T, p, rep, hist, hist_len=None, calls=2):
    B, V = x.shape
    d = {k: rocm.DeviceBuffer.from_numpy(v) if v is not None else None for k, v in dict(x=x, u=u, h=hist, n=hist_len).items()}
    s = rocm.NewSampler(rocm.SamplerConfig(Temperature=T, TopP=p, RepetitionPenalty=rep), max_batch=B, max_vocab=V)
    want = oracle.sample(x, u, T, 0, p, rep, hist, hist_len=hist_len, mode=oracle.MODE_FIXED)
    for _ in range(calls):                                 # (the workspace is left as the next call needs it)
        tok, pr = rocm.DeviceBuffer(4 * B), rocm.DeviceBuffer(4 * B)
        s.Sample(d["x"], B, V, d["h"], d["n"], d["u"], tok, pr, hist_stride=hist.shape[1] if hist is not None else 0)
        s.Status()
        assert np.array_equal(tok.to_numpy(np.int32, (B,)), want["tokens"]), (B, V, T, p, rep)
        assert np.array_equal(pr.to_numpy(np.uint32, (B,)), want["probs"].view(np.uint32)), (B, V, T, p, rep)
    s.Close()


@pytest.mark.parametrize("V", [49151, 49152, 49185, 65536, 100003, 152064, 300001])
@pytest.mark.parametrize("B", [1, 3, 32, 33, 85, 86, 128, 129])
def test_lengths_and_batches(oracle, rocm, B, V):
    rng = np.random.default_rng(V + B)
    if B > 3 and V > 49185:
        B = 5
    x = (2 * rng.standard_normal((B, V))).astype(np.float32)
    u = rng.random(B).astype(np.float32)
    hist = np.concatenate([x.argsort(1)[:, -40:], rng.integers(0, V, (B, 57))], 1).astype(np.int32)
    hist[:, -3:] = [0, V - 1, V // 2]
    hl = rng.integers(0, hist.shape[1] + 1, B).astype(np.int32)
    # (1.9: a temperature whose division has no shortcut in the one-workgroup kernel)
    for T, p, rep, h, n in [(1.0, 1.0, 1.0, None, None), (0.8, 0.95, 1.2, hist, None), (1.9, 0.99, 0.8, hist, hl), (1.3, 0.5, 1.0, hist, None)]:
        _check(oracle, rocm, x, u, T, p, rep, h, n)


@pytest.mark.parametrize("T,p", [(1.0, 1.0), (0.7, 0.9), (1.2, 0.999)])
def test_rows_of_every_kind(oracle, rocm, T, p):
    rng = np.random.default_rng(5)
    V = 70001
    rows = []
    for i in range(4):                                     # a bulk and a few likely tokens: the nucleus is gathered whole, or its draw is told
        x = 1.5 * rng.standard_normal(V)
        x[rng.integers(0, V, 20)] += 6 + 6 * rng.random(20)
        rows.append(x)
    rows.append(np.round(rng.standard_normal(V) * 2) / 2)  # ties by the thousand
    rows.append(np.zeros(V))
    rows.append(np.full(V, -np.inf))
    rows.append(np.where(rng.random(V) < 0.999, -np.inf, rng.standard_normal(V)))
    one = np.full(V, -np.inf)
    one[V - 1] = 3
    rows.append(one)
    wild = rng.standard_normal(V)
    wild[:9] = [np.nan, np.inf, -np.inf, 1e30, -1e30, 1e-40, -0.0, 3e38, -3e38]
    rows.append(wild)
    rows.append(np.where(np.arange(V) % 3 == 0, np.nan, rng.standard_normal(V)))
    rows.append(np.sort(rng.standard_normal(V) * 3))
    rows.append(rng.standard_normal(V) * 1e-3)
    rows.append(rng.standard_normal(V) - 5000)
    x = np.stack(rows).astype(np.float32)
    for seed in range(3):
        u = np.random.default_rng(seed).random(len(x)).astype(np.float32)
        if seed == 2:
            u[:] = np.float32(1 - 2.0 ** -24)
        hist = np.random.default_rng(seed).integers(0, V, (len(x), 300)).astype(np.int32)
        hist[:, :9] = np.arange(9)
        _check(oracle, rocm, x, u, T, p, 1.0, None)
        _check(oracle, rocm, x, u, T, p, 1.3, hist)


@pytest.mark.parametrize("H", [1024, 1025, 4096, 4097])     # 4097: more than the parts' workgroups keep
def test_long_histories(oracle, rocm, H):
    rng = np.random.default_rng(H)
    B, V = 3, 66011
    x = rng.standard_normal((B, V)).astype(np.float32)
    hist = rng.integers(0, V, (B, H)).astype(np.int32)
    hist[1] = 66000 + np.arange(H) % 11                     # all in the last part, the same ids over and over
    _check(oracle, rocm, x, rng.random(B).astype(np.float32), 0.9, 0.9, 1.1, hist)


def test_ids_outside_the_vocabulary_are_reported(rocm):
    V = 65536
    for bad in (-1, -2, V, -2 ** 31, 2 ** 31 - 1):
        x, u, h = np.zeros((2, V), np.float32), np.zeros(2, np.float32), np.full((2, 4), 7, np.int32)
        h[1, 2] = bad
        for rep in (1.0, 1.2):
            s = rocm.NewSampler(rocm.SamplerConfig(RepetitionPenalty=rep), max_batch=2, max_vocab=V)
            tok = rocm.DeviceBuffer(8)
            s.Sample(rocm.DeviceBuffer.from_numpy(x), 2, V, rocm.DeviceBuffer.from_numpy(h), None, rocm.DeviceBuffer.from_numpy(u), tok, None, hist_stride=4)
            with pytest.raises(Exception):
                s.Status()
            s.Close()


def test_captures_before_and_after_the_workspace(oracle, rocm):
    """A handle's first such call under capture (a workgroup to a row: nothing is allocated), then an eager one (which allocates), then one captured
    with the workspace; every replay of either graph, with eager calls between, gives the oracle's."""
    import ctypes as C
    from born_amd import _capi
    hip = C.CDLL("libamdhip64.so")
    rng = np.random.default_rng(6)
    B, V, T, p = 5, 70001, 0.9, 0.95
    xh = (2 * rng.standard_normal((B, V))).astype(np.float32)
    x, u = rocm.DeviceBuffer.from_numpy(xh), rocm.DeviceBuffer(4 * B)
    tok, pr = rocm.DeviceBuffer(4 * B), rocm.DeviceBuffer(4 * B)
    s = rocm.NewSampler(rocm.SamplerConfig(Temperature=T, TopP=p), max_batch=B, max_vocab=V)
    stream = C.c_void_p()
    assert hip.hipStreamCreate(C.byref(stream)) == 0

    def capture():
        graph, graph_exec = C.c_void_p(), C.c_void_p()
        assert hip.hipStreamBeginCapture(stream, 0) == 0
        try:
            s.Sample(x, B, V, None, None, u, tok, pr, stream=stream)
        finally:
            rc = hip.hipStreamEndCapture(stream, C.byref(graph))
        assert rc == 0 and graph.value, "the capture was invalidated"
        assert hip.hipGraphInstantiate(C.byref(graph_exec), graph, None, None, C.c_size_t(0)) == 0
        return graph, graph_exec

    def check(run):
        uh = rng.random(B).astype(np.float32)
        for buf, h in ((u, uh), (tok, np.full(B, -7, np.int32)), (pr, np.full(B, -1, np.float32))):
            _capi.check(_capi.lib().born_rocm_h2d(buf.ptr, h.ctypes.data, h.nbytes, None))
        run()
        assert hip.hipStreamSynchronize(stream) == 0
        s.Status()
        want = oracle.sample(xh, uh, T, 0, p, 1.0, None, mode=oracle.MODE_FIXED)
        assert np.array_equal(tok.to_numpy(np.int32, (B,)), want["tokens"])
        assert np.array_equal(pr.to_numpy(np.uint32, (B,)), want["probs"].view(np.uint32))

    graphs = [capture()]
    replay = lambda g: check(lambda: hip.hipGraphLaunch(g[1], stream))  # noqa: E731
    replay(graphs[0])
    eager = lambda: check(lambda: s.Sample(x, B, V, None, None, u, tok, pr, stream=stream))  # noqa: E731
    eager()
    graphs.append(capture())
    for _ in range(3):
        for g in graphs:
            replay(g)
            eager()
    for graph, graph_exec in graphs:
        hip.hipGraphExecDestroy(graph_exec)
        hip.hipGraphDestroy(graph)
    hip.hipStreamDestroy(stream)
    s.Close()
