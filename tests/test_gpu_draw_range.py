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


@pytest.mark.parametrize("B,V", [(8, 50257), (300, 28676), (3, 100003)])    # 1024 and 512 threads to a row; rows in parts
def test_logits_without_mass_do_not_queue(oracle, B, V):
    """Rows of a mask that leaves one logit in ten, and rows of one logit far above the others: what lies beyond the bins of masses is added up apart, so that they take no
    longer than rows of a model (2.2 times as long where all of it was added to one bin, and longer the longer the row)."""
    import time

    from born_amd import sampler as S
    rng = np.random.default_rng(V)
    plain = (2 * rng.standard_normal((B, V))).astype(np.float32)
    masked = np.where(rng.random((B, V)) < 0.9, np.float32(-np.inf), plain)
    peak = plain.copy()
    peak[:, V // 2] += 60
    u = rng.random(B).astype(np.float32)
    for T in (1.0, 0.7):
        s = S.NewSampler(S.SamplerConfig(Temperature=T, TopP=0.95), max_batch=B, max_vocab=V)
        du, tok, prob = S.DeviceBuffer.from_numpy(u), S.DeviceBuffer(4 * B), S.DeviceBuffer(4 * B)
        took = []
        for x in (plain, masked, peak):
            dx = S.DeviceBuffer.from_numpy(x)
            best = np.inf
            for _ in range(12):
                s.Status()                                  # (waits)
                t0 = time.perf_counter()
                for _ in range(40):
                    s.Sample(dx, B, V, None, None, du, tok, prob)
                s.Status()
                best = min(best, time.perf_counter() - t0)
            took.append(best)
            want = oracle.sample(x[:4], u[:4], T, 0, 0.95, 1.0, None, mode=oracle.MODE_FIXED)
            assert np.array_equal(tok.to_numpy(np.int32, (B,))[:4], want["tokens"])
            assert np.array_equal(prob.to_numpy(np.uint32, (B,))[:4], want["probs"].view(np.uint32))
        s.Close()
        assert max(took[1:]) <= 1.5 * took[0], took


@pytest.mark.parametrize("offset", [0, 5, -50, 30000])
@pytest.mark.parametrize("spread", [1e-6, 1e-3, 0.01, 1])
def test_logits_that_hardly_differ(oracle, spread, offset):
    """Bins as narrow as a few roundings of what is compared with their bounds; in one workgroup of 1024 and 512 threads, and in parts."""
    from born_amd import sampler as S
    rng = np.random.default_rng(abs(offset) + 1)
    for B, V, path in ((6, 8193, 0), (6, 20001, 2), (2, 70001, 0)):
        x = (spread * rng.standard_normal((B, V)) + offset).astype(np.float32)
        u, hist = rng.random(B).astype(np.float32), rng.integers(0, V, (B, 30)).astype(np.int32)
        for T, p, rep in ((1.0, 0.6, 1.0), (0.7, 0.95, 1.0001), (1.9, 0.999, 1.0), (1.3, 1.0, 1.2)):
            s = S.NewSampler(S.SamplerConfig(Temperature=T, TopP=p, RepetitionPenalty=rep), max_batch=B, max_vocab=V)
            s.SetPath(path)
            got = S.sample_host(s, x, u, hist)
            s.Status()
            s.Close()
            want = oracle.sample(x, u, T, 0, p, rep, hist, mode=oracle.MODE_FIXED)
            assert np.array_equal(got["tokens"], want["tokens"]), (B, V, T, p)
            assert np.array_equal(got["probs"].view(np.uint32), want["probs"].view(np.uint32)), (B, V, T, p)


def test_logits_that_hardly_differ_take_no_longer(oracle):
    """128 rows of 152 064 logits of a spread of 0.01, whose bins are a fifth of 1e-4 wide: four times as long as rows of a model while that much was
    gathered beside the wanted bins, more than the lists hold."""
    import time

    from born_amd import sampler as S
    rng = np.random.default_rng(3)
    B, V, T, p = 128, 152064, 1.0, 0.6
    plain = (2 * rng.standard_normal((B, V))).astype(np.float32)
    u = rng.random(B).astype(np.float32)
    s = S.NewSampler(S.SamplerConfig(Temperature=T, TopP=p), max_batch=B, max_vocab=V)
    du, tok, prob = S.DeviceBuffer.from_numpy(u), S.DeviceBuffer(4 * B), S.DeviceBuffer(4 * B)
    took = []
    for x in (plain, plain * np.float32(0.005)):
        dx = S.DeviceBuffer.from_numpy(x)
        best = np.inf
        for _ in range(12):
            s.Status()                                      # (waits)
            t0 = time.perf_counter()
            for _ in range(20):
                s.Sample(dx, B, V, None, None, du, tok, prob)
            s.Status()
            best = min(best, time.perf_counter() - t0)
        took.append(best)
        want = oracle.sample(x[:3], u[:3], T, 0, p, 1.0, None, mode=oracle.MODE_FIXED)
        assert np.array_equal(tok.to_numpy(np.int32, (B,))[:3], want["tokens"])
        assert np.array_equal(prob.to_numpy(np.uint32, (B,))[:3], want["probs"].view(np.uint32))
    s.Close()
    assert took[1] <= 2 * took[0], took
