"""Rows that start at any four bytes (a vocabulary that is no multiple of four) under 128-bit loads: the row's last one to three
logits, and the ends of the kernels' stages (8192 and 16384 logits), against the oracle's fixed-point layer, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LENGTHS = [3, 4, 5, 6, 7, 8191, 8193, 16381, 16383, 16385, 24575, 32766, 32769, 49151, 49154, 65537, 81923]


@pytest.fixture(scope="module")
def rocm():
    from born_amd import sampler as S
    assert S.DeviceCount() >= 1, "no HIP device visible"
    return S


def _rows(V, B=7):
    rng = np.random.default_rng(V)
    x = rng.standard_normal((B, V)).astype(np.float32)
    x[1::2, V - 3:] += np.float32(6)                       # every other row's likely tokens are its very last ones
    x[2, V - 1], x[4, V - 2] = np.nan, -np.inf
    return x, rng.random(B).astype(np.float32)


@pytest.mark.parametrize("path", [0, 2])                   # 2: 512 threads to a row, whatever the batch
@pytest.mark.parametrize("k,p,T", [(3, 1.0, 1.0), (50, 0.9, 0.7), (0, 0.95, 0.7), (0, 1.0, 1.0)])
@pytest.mark.parametrize("V", LENGTHS)
def test_sampling(oracle, rocm, V, k, p, T, path):
    x, u = _rows(V)
    hist = np.tile(np.array([[V - 1, 0, V - 3]], np.int32), (len(x), 1))
    s = rocm.NewSampler(rocm.SamplerConfig(Temperature=T, TopK=min(k, V), TopP=p, RepetitionPenalty=1.2), max_batch=len(x), max_vocab=V)
    s.SetPath(path)
    got = rocm.sample_host(s, x, u, hist)
    s.Status()
    s.Close()
    want = oracle.sample(x, u, T, min(k, V), p, 1.2, hist, mode=oracle.MODE_FIXED)
    assert np.array_equal(got["tokens"], want["tokens"])
    assert np.array_equal(got["probs"].view(np.uint32), want["probs"].view(np.uint32))


@pytest.mark.parametrize("T", [1.0, 0.8])
@pytest.mark.parametrize("V", [3, 5, 4095, 4097, 32765, 32767, 32771])
def test_verification(oracle, rocm, V, T):
    rng = np.random.default_rng(V)
    B, G = 5, 2
    t = rng.standard_normal((B, G, V)).astype(np.float32)
    d = (t + rng.standard_normal((B, G, V))).astype(np.float32)
    t[::2, :, V - 2:] += np.float32(4)
    d[0, 0, V - 1] = np.nan
    tok = rng.integers(0, V, (B, G)).astype(np.int32)
    tok[1:3] = V - 1
    ua, ur = rng.random((B, G)).astype(np.float32), rng.random(B).astype(np.float32)
    s = rocm.NewSampler(rocm.SamplerConfig(Temperature=T), max_batch=B, max_vocab=V)
    got = rocm.verify_host(s, t, d, tok, ua, ur)
    s.Status()
    s.Close()
    want = oracle.spec_verify(t, d, tok, ua, ur, temperature=T, mode=oracle.MODE_FIXED)
    assert np.array_equal(got["n_accepted"], want["n_accepted"]) and np.array_equal(got["next_token"], want["next_token"])
