"""Linear layers over a handful of rows: one to five rows (the last is the tiles'), columns around the groups of four and where a
workgroup shares them, K around a load, a stage and the quarters of K, against fp64.  A result is a chain of at most K / 64 + 4 fused
multiply-adds a lane, six pairwise additions, three more over the quarters of K, and the bias."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mods():
    from born_amd import linear, sampler
    return linear, sampler


def _layer(mods, rng, K, N):
    L, S = mods
    w, b = rng.standard_normal((N, K)).astype(np.float32), rng.standard_normal(N).astype(np.float32)
    return w, b, L.Linear(K, N, S.DeviceBuffer.from_numpy(w), S.DeviceBuffer.from_numpy(b))


@pytest.mark.parametrize("K", [4, 8, 252, 256, 260, 508, 512, 516, 1024, 1028, 2052, 4096])
@pytest.mark.parametrize("N", [1, 3, 4, 5, 1001, 8191, 8192, 8197])
def test_against_fp64(mods, K, N):
    L, S = mods
    rng = np.random.default_rng(K * N)
    w, b, layer = _layer(mods, rng, K, N)
    x = rng.standard_normal((4, K)).astype(np.float32)
    exact = x.astype(np.float64) @ w.T.astype(np.float64) + b
    chain = K / 64 + 14 if N < 8192 or K >= 1024 else K + 4     # (more than one row of a short K and many columns: the tiles' chains)
    bound = chain * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w).T.astype(np.float64) + np.abs(b))
    for M in range(1, 5):
        out = S.DeviceBuffer(4 * M * N)
        layer.Forward(S.DeviceBuffer.from_numpy(x[:M]), (M, K), out)
        assert (np.abs(out.to_numpy(np.float32, (M, N)) - exact[:M]) <= bound[:M]).all(), M


@pytest.mark.parametrize("M", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("K,N", [(260, 5000), (512, 20003), (4096, 8200)])
def test_the_greedy_token_is_the_plain_head_s(oracle, mods, M, K, N):
    L, S = mods
    rng = np.random.default_rng(M)
    w, b, layer = _layer(mods, rng, K, N)
    x = S.DeviceBuffer.from_numpy(rng.standard_normal((M, K)).astype(np.float32))
    out, tok = S.DeviceBuffer(4 * M * N), S.DeviceBuffer(4 * M)
    layer.Forward(x, (M, K), out)
    logits = out.to_numpy(np.float32, (M, N))
    s = S.NewSampler(S.SamplerConfig(Temperature=0.8, TopK=20, TopP=0.9), max_batch=M, max_vocab=N)
    L.ForwardArgmax(s, layer, x, (M, K), tok)
    assert np.array_equal(tok.to_numpy(np.int32, (M,)), logits.argmax(-1))
    # head and sampling step in one call draw from these very logits
    u = rng.random(M).astype(np.float32)
    tokens, probs, _ = L.ForwardSampleHost(s, layer, x, (M, K), None, None, S.DeviceBuffer.from_numpy(u))
    want = oracle.sample(logits, u, 0.8, 20, 0.9, 1.0, None, mode=oracle.MODE_FIXED)
    assert np.array_equal(tokens, want["tokens"]) and np.array_equal(probs.view(np.uint32), want["probs"].view(np.uint32))
    s.Close()


def test_what_is_not_finite_stays_in_its_row_and_column(mods):
    L, S = mods
    rng = np.random.default_rng(1)
    M, K, N = 4, 772, 9001                                   # (a stage that is not whole)
    w, b, _ = _layer(mods, rng, K, N)
    x = rng.standard_normal((M, K)).astype(np.float32)
    w[7, K - 1], w[8, 0], x[2, K - 1] = np.inf, np.nan, -np.inf
    out = S.DeviceBuffer(4 * M * N)
    L.Linear(K, N, S.DeviceBuffer.from_numpy(w), S.DeviceBuffer.from_numpy(b)).Forward(S.DeviceBuffer.from_numpy(x), (M, K), out)
    got = out.to_numpy(np.float32, (M, N))
    with np.errstate(invalid="ignore"):
        exact = x.astype(np.float64) @ w.T.astype(np.float64) + b
    assert np.array_equal(np.isnan(got), np.isnan(exact)) and np.array_equal(np.isposinf(got), np.isposinf(exact))
    ok = np.isfinite(exact)
    assert np.allclose(got[ok], exact[ok], rtol=0, atol=1e-3)


@pytest.mark.parametrize("M,K,N", [(1, 32, 16383), (1, 32, 16384), (1, 188, 24575), (1, 44, 24577), (1, 52, 24577), (1, 192, 16400), (1, 160, 16400), (1, 288, 40001),
                                   (1, 320, 40001), (3, 1024, 24577), (4, 3068, 24580), (4, 3072, 24580), (3, 1024, 32769), (2, 1024, 30000)])
def test_either_side_of_the_lines(mods, M, K, N):
    """Where one row, or three and four, of many columns pass from the tiles to the waves: a chain of K at most, and the bias."""
    L, S = mods
    rng = np.random.default_rng(K + N)
    w, b, layer = _layer(mods, rng, K, N)
    x = rng.standard_normal((M, K)).astype(np.float32)
    out = S.DeviceBuffer(4 * M * N)
    layer.Forward(S.DeviceBuffer.from_numpy(x), (M, K), out)
    exact = x.astype(np.float64) @ w.T.astype(np.float64) + b
    bound = (K + 4) * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w).T.astype(np.float64) + np.abs(b))
    assert (np.abs(out.to_numpy(np.float32, (M, N)) - exact) <= bound).all()
