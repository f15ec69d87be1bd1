"""Rows without a top-k cut whose wanted bins hold equal logits: lists around the 32 entries that are summed directly, the 1024 or 512 that fit, and beyond;
rows around the 1024 logits from which a bin's masses are added in fp64; rows in parts.  Against the oracle's fixed-point layer, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("path", [0, 2])                    # 2: 512 threads to a row
@pytest.mark.parametrize("p", [0.6, 1.0])
@pytest.mark.parametrize("V,ties", [(1023, 31), (1023, 33), (1024, 32), (1056, 33), (2048, 128), (8193, 129), (16400, 511), (16400, 513), (30000, 1023), (40001, 1025),
                                    (66001, 300), (66001, 1100)])
def test_lists_of_equal_logits(oracle, V, ties, p, path):
    from born_amd import sampler as S
    rng = np.random.default_rng(V + ties)
    B = 6
    levels = -(-V // ties)
    values = np.sort(rng.standard_normal(levels)).astype(np.float32)
    x = np.stack([rng.permutation(values[np.arange(V) // ties]) for _ in range(B)])
    x[1] *= 0.01                                            # masses that hardly differ
    x[2, rng.choice(V, V // 2, replace=False)] = -np.inf
    x[3] += 1e-4 * rng.standard_normal(V).astype(np.float32)  # nearly equal: many entries to a bucket, or many buckets
    u = rng.random(B).astype(np.float32)
    u[0], u[4] = 0, 1 - 2.0 ** -24
    hist = rng.integers(0, V, (B, 40)).astype(np.int32)
    for T, rep in ((1.0, 1.0), (0.7, 1.3)):
        s = S.NewSampler(S.SamplerConfig(Temperature=T, TopP=p, RepetitionPenalty=rep), max_batch=B, max_vocab=V)
        s.SetPath(path)
        got = S.sample_host(s, x, u, hist)
        s.Status()
        s.Close()
        want = oracle.sample(x, u, T, 0, p, rep, hist, mode=oracle.MODE_FIXED)
        assert np.array_equal(got["tokens"], want["tokens"])
        assert np.array_equal(got["probs"].view(np.uint32), want["probs"].view(np.uint32))


@pytest.mark.parametrize("B,V", [(3, 54165), (3, 54166), (32, 57141), (32, 57142), (42, 59998), (42, 59999), (51, 74998), (51, 74999), (64, 79998), (64, 79999), (85, 89998), (85, 89999),
                                 (128, 196607), (128, 196608)])
def test_rows_around_the_shortest_that_are_cut(oracle, B, V):
    """The sizes of tests/test_nucleus_plan.py, which holds that one of each pair is cut."""
    from born_amd import sampler as S
    rng = np.random.default_rng(B + V)
    x = (2 * rng.standard_normal((4, V))).astype(np.float32)
    x = np.concatenate([x] * (B // 4 + 1))[:B]
    u = rng.random(B).astype(np.float32)
    s = S.NewSampler(S.SamplerConfig(Temperature=0.8, TopP=0.95), max_batch=B, max_vocab=V)
    got = S.sample_host(s, x, u, None)
    s.Status()
    s.Close()
    at = [0, 1, 2, B // 2, B - 1]
    want = oracle.sample(x[at], u[at], 0.8, 0, 0.95, 1.0, None, mode=oracle.MODE_FIXED)
    assert np.array_equal(got["tokens"][at], want["tokens"])
    assert np.array_equal(got["probs"][at].view(np.uint32), want["probs"].view(np.uint32))


@pytest.mark.parametrize("B,V,step,T,p", [(32, 50257, 30, 0.8, 0.95), (32, 50257, 30, 1.9, 0.9), (200, 32000, 30, 1.9, 0.9), (512, 8191, 3, 1.0, 0.6), (512, 2048, 3, 1.9, 0.9)])
def test_levels_of_which_one_fits_the_list(oracle, B, V, step, T, p):
    """Logits of a few hundred equal ones each: where the cut's fit the lists but not the draw's beside them, the cut's are listed: no row is left to the descent for both."""
    from born_amd import sampler as S
    rng = np.random.default_rng(V)
    x = (np.round(step * rng.standard_normal((B, V))) * (2 / step)).astype(np.float32)
    u = rng.random(B).astype(np.float32)
    s = S.NewSampler(S.SamplerConfig(Temperature=T, TopP=p), max_batch=B, max_vocab=V)
    got = S.sample_host(s, x, u, None)
    s.Status()
    counters = s.Counters()
    s.Close()
    want = oracle.sample(x, u, T, 0, p, 1.0, None, mode=oracle.MODE_FIXED)
    assert np.array_equal(got["tokens"], want["tokens"])
    assert np.array_equal(got["probs"].view(np.uint32), want["probs"].view(np.uint32))
    assert counters["fallback_rows"] == 0, counters
