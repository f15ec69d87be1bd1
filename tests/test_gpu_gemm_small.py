"""Small products: rows, columns and K around a square, a chunk and the waves' shares of K, the squares of 16 and of 32, operands of any start
and pitch with NaNs around them, the plain and the fused forms, against fp64 with the tolerance of the fp32 products:
(4 sqrt(K) + 2) 2^-24 (|a| |b| + |bias|)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(M, K, N) for M in (1, 5, 16, 17) for K in (1, 3, 16, 63, 64, 65, 127, 255, 257, 513, 1000) for N in (1, 15, 16, 17, 33)] + [
    (64, 784, 512), (64, 1024, 128), (160, 340, 1024), (160, 341, 960), (160, 344, 961), (335, 65, 641), (336, 64, 641), (336, 300, 656), (37, 1000, 1500),
    (33, 2100, 65), (1001, 63, 100), (4096, 32, 10), (2100, 96, 64), (128, 2048, 256), (16, 2080, 2048)]


def _placed(S, a, before, over):
    """a at a pitch of its columns + over, `before` floats into a buffer of NaNs."""
    rows, cols = a.shape
    flat = np.full(before + rows * (cols + over) + 8, np.nan, np.float32)
    flat[before:before + rows * (cols + over)].reshape(rows, cols + over)[:, :cols] = a
    buf = S.DeviceBuffer.from_numpy(flat)
    return buf, buf.ptr + 4 * before, cols + over


@pytest.mark.parametrize("before,over", [(0, 0), (4, 8), (1, 3)])
def test_against_fp64(before, over):
    from born_amd import _capi, sampler as S
    for i, (M, K, N) in enumerate(SHAPES):
        rng = np.random.default_rng(i)
        x, w, b = (rng.standard_normal(s).astype(np.float32) for s in ((M, K), (N, K), (1, N)))
        exact = x.astype(np.float64) @ w.T.astype(np.float64)
        mag = np.abs(x).astype(np.float64) @ np.abs(w).T.astype(np.float64)
        keep = [_placed(S, a, before, over) for a in (x, w, np.ascontiguousarray(w.T), b)]
        (_, px, lx), (_, pw, lw), (_, pt, lt), (_, pb, _) = keep
        for form in ("linear", "matmul"):
            out = S.DeviceBuffer.from_numpy(np.full((M, N + over), 7, np.float32))
            if form == "linear":
                _capi.check(_capi.lib().born_rocm_linear(px, M, K, lx, pw, N, lw, pb, out.ptr, N + over, None))
                want, tol = exact + b, mag + np.abs(b)
            else:
                _capi.check(_capi.lib().born_rocm_matmul(px, pt, out.ptr, M, K, N, lx, lt, N + over, None))
                want, tol = exact, mag
            got = out.to_numpy(np.float32, (M, N + over))
            assert (np.abs(got[:, :N] - want) <= (4 * np.sqrt(K) + 2) * 2.0 ** -24 * tol).all(), (form, M, K, N)
            assert (got[:, N:] == 7).all(), (form, M, K, N)


@pytest.mark.parametrize("M,K,N", [(64, 2048, 1024), (497, 1568, 232), (94, 3212, 101), (2000, 2000, 100), (400, 4097, 300), (911, 19590, 17), (3, 30001, 700)])
def test_error_of_a_sum_in_sixteen_parts(M, K, N):
    """No sum of the product is longer than K / 16 terms, as in the tiles' most slices.  A sum of L terms that are alike grows as sqrt(j), each addition rounds by
    2^-24 / sqrt(3) of it at most, root mean square, so that sqrt(L / 6) 2^-24 is the most of a part's, and of the whole, 2-norm."""
    from born_amd import _capi, sampler as S
    rng = np.random.default_rng(K)
    x, w = rng.standard_normal((M, K)).astype(np.float32), rng.standard_normal((N, K)).astype(np.float32)
    exact = x.astype(np.float64) @ w.T.astype(np.float64)
    px, pw, pt, out = S.DeviceBuffer.from_numpy(x), S.DeviceBuffer.from_numpy(w), S.DeviceBuffer.from_numpy(np.ascontiguousarray(w.T)), S.DeviceBuffer(4 * M * N)
    for form in ("linear", "matmul"):
        if form == "linear":
            _capi.check(_capi.lib().born_rocm_linear(px.ptr, M, K, K, pw.ptr, N, K, None, out.ptr, N, None))
        else:
            _capi.check(_capi.lib().born_rocm_matmul(px.ptr, pt.ptr, out.ptr, M, K, N, K, N, N, None))
        err = np.linalg.norm(out.to_numpy(np.float32, (M, N)) - exact) / np.linalg.norm(exact)
        assert err <= np.sqrt(K / 16 / 6) * 2.0 ** -24, (form, err)


@pytest.mark.parametrize("M,K,N", [(5, 300, 300), (17, 256, 1001), (33, 352, 5000), (64, 1024, 200)])
def test_the_fused_heads_see_the_plain_head_s_logits(oracle, M, K, N):
    from born_amd import linear as L, sampler as S
    rng = np.random.default_rng(M)
    w, b = (rng.standard_normal((N, K)) * 2 / np.sqrt(K)).astype(np.float32), rng.standard_normal(N).astype(np.float32)
    layer = L.Linear(K, N, S.DeviceBuffer.from_numpy(w), S.DeviceBuffer.from_numpy(b))
    x = S.DeviceBuffer.from_numpy(rng.standard_normal((M, K)).astype(np.float32))
    out, tok = S.DeviceBuffer(4 * M * N), S.DeviceBuffer(4 * M)
    layer.Forward(x, (M, K), out)
    logits = out.to_numpy(np.float32, (M, N))
    s = S.NewSampler(S.SamplerConfig(Temperature=0.8, TopK=20, TopP=0.9), max_batch=M, max_vocab=N)
    L.ForwardArgmax(s, layer, x, (M, K), tok)
    assert np.array_equal(tok.to_numpy(np.int32, (M,)), logits.argmax(-1))
    u = rng.random(M).astype(np.float32)
    tokens, probs, _ = L.ForwardSampleHost(s, layer, x, (M, K), None, None, S.DeviceBuffer.from_numpy(u))
    want = oracle.sample(logits, u, 0.8, 20, 0.9, 1.0, None, mode=oracle.MODE_FIXED)
    assert np.array_equal(tokens, want["tokens"]) and np.array_equal(probs.view(np.uint32), want["probs"].view(np.uint32))
    s.Close()
