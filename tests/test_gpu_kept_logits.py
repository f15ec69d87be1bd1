"""Sampling without a top-k cut: rows around the lengths from which their first logits stay in registers between the sweeps, and where what stays is all
of them; aligned and ragged, with and without a history, whose ids fall into what stays and beyond it.  Against the oracle's fixed-point layer, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _check(oracle, B, V, path, at):
    from born_amd import sampler as S
    rng = np.random.default_rng(V + B)
    x = (2 * rng.standard_normal((B, V))).astype(np.float32)
    if B > 2:
        x[1, rng.integers(0, V, 20)] += 8
        x[2, ::3] = -np.inf
    u = rng.random(B).astype(np.float32)
    hist = np.concatenate([x.argsort(1)[:, -20:], rng.integers(0, V, (B, 200))], 1).astype(np.int32)
    hist[:, -4:] = [0, V - 1, min(V - 1, 16384), min(V - 1, 20480)]
    for T, p, rep, h in ((1.0, 1.0, 1.0, None), (0.8, 0.95, 1.2, hist), (1.3, 0.5, 1.0, None), (1.9, 0.9, 0.8, hist)):   # (1.9: no shortcut for its division)
        s = S.NewSampler(S.SamplerConfig(Temperature=T, TopP=p, RepetitionPenalty=rep), max_batch=B, max_vocab=V)
        s.SetPath(path)
        got = S.sample_host(s, x, u, h)
        s.Status()
        s.Close()
        want = oracle.sample(x[at], u[at], T, 0, p, rep, None if h is None else h[at], mode=oracle.MODE_FIXED)
        assert np.array_equal(got["tokens"][at], want["tokens"]), (T, p)
        assert np.array_equal(got["probs"][at].view(np.uint32), want["probs"].view(np.uint32)), (T, p)


@pytest.mark.parametrize("V", [28667, 28668, 28671, 28672, 28673, 28675, 28676, 30720, 36863, 36864, 36868])
def test_two_rows_to_a_cu(oracle, V):
    """Ten blocks of a thread stay from fourteen on: 28 672 logits; the loop's two stages of four blocks of 512 threads turn at 8192 more."""
    _check(oracle, 5, V, 2, [0, 1, 2, 3, 4])


@pytest.mark.parametrize("V", [16385, 16387, 16388, 20000, 32768, 32771, 32772])
def test_a_row_to_a_cu(oracle, V):
    """A stage of four blocks of 1024 threads stays, 16 384 logits, in batches beyond 16 MiB."""
    _check(oracle, 256, V, 0, [0, 1, 2, 100, 255])


@pytest.mark.parametrize("V", [3, 1535, 4095, 16383, 16384, 16385, 28671, 28672, 32769])
@pytest.mark.parametrize("B", [6, 300])
def test_rows_with_settings_of_their_own(oracle, B, V):
    """Those keep at every length."""
    from born_amd import sampler as S
    rng = np.random.default_rng(V)
    x = (2 * rng.standard_normal((B, V))).astype(np.float32)
    u, hist = rng.random(B).astype(np.float32), rng.integers(0, V, (B, 50)).astype(np.int32)
    T, p, rep = (0.6 + 0.9 * rng.random(B)).astype(np.float32), (0.5 + 0.5 * rng.random(B)).astype(np.float32), (1 + 0.3 * rng.random(B)).astype(np.float32)
    k = np.zeros(B, np.int32)
    d = {n: S.DeviceBuffer.from_numpy(a) for n, a in dict(x=x, u=u, h=hist, T=T, p=p, rep=rep, k=k).items()}
    tok, pr = S.DeviceBuffer(4 * B), S.DeviceBuffer(4 * B)
    s = S.NewSampler(S.SamplerConfig(), max_batch=B, max_vocab=V)
    s.SampleRows(d["x"], B, V, d["h"], None, d["u"], d["T"], d["k"], d["p"], d["rep"], tok, pr, hist_stride=50)
    s.Status()
    s.Close()
    tokens, probs = tok.to_numpy(np.int32, (B,)), pr.to_numpy(np.uint32, (B,))
    for b in {0, 1, B // 2, B - 1}:
        want = oracle.sample(x[b:b + 1], u[b:b + 1], float(T[b]), 0, float(p[b]), float(rep[b]), hist[b:b + 1], mode=oracle.MODE_FIXED)
        assert tokens[b] == want["tokens"][0] and probs[b] == want["probs"].view(np.uint32)[0], b
