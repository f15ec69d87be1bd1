"""Top-p without a top-k cut: the draw among the bins that the mass of the nucleus allows, one or many of them, next to the cut's bin, in it or
far above.  Short rows (most bins empty, each logit a large share), rows of a bulk and a few likely tokens, and uniforms at both ends, against
the oracle's fixed-point layer, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("path", [0, 2])                    # 2: 512 threads to a row
@pytest.mark.parametrize("p", [0.3, 0.9, 0.99])
@pytest.mark.parametrize("V", [2, 65, 300, 1001, 8193, 40000])
def test_draws(oracle, V, p, path):
    from born_amd import sampler as S
    rng = np.random.default_rng(V + int(100 * p))
    B = 48
    x = (1.5 * rng.standard_normal((B, V))).astype(np.float32)
    for b in range(0, B, 2):                                # a few likely tokens over the bulk
        at = rng.choice(V, min(V, 1 + b), replace=False)
        x[b, at] += rng.uniform(2, 10, at.size).astype(np.float32)
    x[5] = x[5, 0]                                          # nothing but ties
    x[7, V // 2:] = -np.inf
    u = rng.random(B).astype(np.float32)
    u[0], u[1], u[2], u[3] = 0, 0, 1 - 2.0 ** -24, 1 - 2.0 ** -24
    hist = rng.integers(0, V, (B, 16)).astype(np.int32)
    s = S.NewSampler(S.SamplerConfig(Temperature=0.8, TopP=p, RepetitionPenalty=1.2), max_batch=B, max_vocab=V)
    s.SetPath(path)
    got = S.sample_host(s, x, u, hist)
    s.Status()
    s.Close()
    want = oracle.sample(x, u, 0.8, 0, p, 1.2, hist, mode=oracle.MODE_FIXED)
    assert np.array_equal(got["tokens"], want["tokens"])
    assert np.array_equal(got["probs"].view(np.uint32), want["probs"].view(np.uint32))
