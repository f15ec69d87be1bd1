"""The large products on the 16-bit matrix cores (born_amd/csrc/gemm_split.hip) against fp64 products: every tile and load
form at the edges of tiles and of K, slices of K, rows in chunks, and operands the parts cannot hold.  (What two fp16 parts, K of 256 and more, lose
and when: tests/test_gpu_gemm_f16_parts.py.)

Tolerance: that of tests/test_gpu_linear.py, (4 sqrt(K) + 2) 2^-24 (sum |a| |b| + |bias|).  Three rounded bf16 parts hold an fp32
value exactly and what the six products leave out is at most about 2^-24 |a b| a product, one of the bound's 4 sqrt(K) + 2 units; two fp16 parts take
eight.  Integer-valued operands of up to 22 bits whose partial sums stay below 2^24 are exact.
"""
import numpy as np
import pytest

from tests.test_gpu_linear import EPS, _bound, _gpu_linear, _gpu_matmul, lin, rocm  # noqa: F401  (fixtures)

pytestmark = pytest.mark.gpu

# at least 3 GFLOP and more than 32 rows: what is routed there.  Tiles of 64 x 128, 128 x 128, 128 x 256 and 256 x 256; M, N at
# one past and one short of a tile; K of every load form (a multiple of 64, of 32, of 4, odd) and shorter than a group pair
SHAPES = [(33, 46000, 1024), (64, 8193, 3000), (65, 33000, 800), (129, 40001, 304), (127, 6000, 2055), (257, 50000, 160),
          (256, 100001, 61), (500, 3100, 1000), (200, 2047, 4096), (300, 21539, 288), (1030, 1500, 1028)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("form", ["linear", "matmul"])
def test_matches_fp64(rocm, lin, shape, form):  # noqa: F811
    M, N, K = shape
    rng = np.random.default_rng(M * 7 + N * 3 + K)
    x = rng.standard_normal((M, K), dtype=np.float32)
    w = rng.standard_normal((N, K), dtype=np.float32)
    bias = rng.standard_normal(N, dtype=np.float32) if form == "linear" else None
    got = _gpu_linear(rocm, lin, x, w, bias) if form == "linear" else _gpu_matmul(rocm, lin, x, np.ascontiguousarray(w.T))
    exact = x.astype(np.float64) @ w.T.astype(np.float64) + (0 if bias is None else bias[None, :])
    err = np.abs(got - exact) / _bound(x, w, bias, K)
    assert err.max() <= 1.0, f"{shape}: off the fp64 product by {err.max():.2f} bounds"
    # and no further off, overall, than a product of fp32 sums in blocks of two: half the ulps of sqrt(K / 2) additions
    rms = np.sqrt(np.mean((got - exact) ** 2) / np.mean(exact ** 2))
    assert rms <= 0.5 * np.sqrt(K / 2) * EPS + EPS, (shape, rms)


WORST = np.float32(1 + 2.0 ** -8 - 2.0 ** -17)            # bf16 parts 1, 2^-8, -2^-17: what three leave out of its square is the most


def _operand(rng, family, rows, K):
    if family == "positive":
        return rng.random((rows, K), dtype=np.float32) + np.float32(0.5)
    if family == "equal":
        return np.full((rows, K), WORST)
    if family == "equal, signed":
        return WORST * rng.choice(np.array([-1, 1], np.float32), (rows, K))
    x = rng.standard_normal((rows, K), dtype=np.float32)
    return np.ldexp(x, rng.integers(-10, 11, (rows, K))).astype(np.float32) if family == "magnitudes" else x


@pytest.mark.parametrize("K", [16, 64, 1000, 4096])
@pytest.mark.parametrize("family", ["normal", "positive", "equal", "equal, signed", "magnitudes"])
def test_error_is_no_larger_than_the_fp32_tiles(rocm, lin, family, K):  # noqa: F811
    """The 2-norm of the error against fp64, beside that of the same rows 32 at a time, which the fp32 tiles multiply.  Two correct sums
    of tens of thousands of results: 3 % for the sample."""
    M = 64
    N = int(3.05e9 / (2 * M * K))
    rng = np.random.default_rng(K)
    x, w = _operand(rng, family, M, K), _operand(rng, family, N, K)
    layer, dx = lin.Linear(K, N, rocm.DeviceBuffer.from_numpy(w), None), rocm.DeviceBuffer.from_numpy(x)
    one, two = rocm.DeviceBuffer(M * N * 4), rocm.DeviceBuffer(M * N * 4)
    layer.Forward(dx, (M, K), one)
    for r in (0, 32):
        layer.Forward(dx.ptr + 4 * r * K, (32, K), two.ptr + 4 * r * N)
    some = rng.choice(N, min(N, 2000), replace=False)
    exact = x.astype(np.float64) @ w[some].T.astype(np.float64)
    split, tiles = (np.sqrt(np.mean((b.to_numpy(np.float32, (M, N))[:, some] - exact) ** 2)) for b in (one, two))
    assert split <= 1.03 * tiles, (split, tiles)


@pytest.mark.parametrize("shape", [(70, 24000, 960), (300, 21539, 288)])
def test_integer_valued_operands_are_exact(rocm, lin, shape):  # noqa: F811
    M, N, K = shape
    rng = np.random.default_rng(5)
    x = rng.integers(-100, 101, (M, K)).astype(np.float32)
    w = rng.integers(-100, 101, (N, K)).astype(np.float32)
    x[:, ::17] *= 513                                    # values that take two and three bf16 parts (two fp16 parts'); every sum stays below 2^24
    x[:, 1::3] = 0
    w[:, ::17] = np.sign(w[:, ::17])
    want = x.astype(np.float64) @ w.T.astype(np.float64)
    assert np.abs(x).astype(np.float64).__matmul__(np.abs(w).T.astype(np.float64)).max() < 2.0 ** 24
    assert np.array_equal(_gpu_linear(rocm, lin, x, w, None), want.astype(np.float32))
    assert np.array_equal(_gpu_matmul(rocm, lin, x, np.ascontiguousarray(w.T)), want.astype(np.float32))


@pytest.mark.parametrize("shape", [(200, 8272, 1056), (128, 4096, 4096), (80, 20000, 1024)])
def test_operands_the_parts_cannot_hold(rocm, lin, shape):  # noqa: F811
    """Infinities, NaN, values next to the largest float, and magnitudes whose low parts leave bf16's range, in either
    operand: what an fp32 product gives."""
    M, N, K = shape
    rng = np.random.default_rng(17)
    x = rng.standard_normal((M, K), dtype=np.float32)
    w = rng.standard_normal((N, K), dtype=np.float32)
    x[3, 5], x[40, 7], x[M - 1, K - 1] = np.inf, np.nan, -np.inf
    x[9, :], x[9, 4] = 0.0, np.float32(3.4e38)           # alone in its row: no overflow
    w[:, 4], x[:, K - 2] = np.clip(w[:, 4], -0.9, 0.9), np.clip(x[:, K - 2], -0.9, 0.9)
    w[17, 30], w[N - 1, 2], w[130, K - 2] = np.inf, np.nan, np.float32(-3.4e38)
    x[50, :] *= np.float32(2.0 ** -120)                  # a row of tiny values ..
    w[200, :] *= np.float32(2.0 ** 90)                   # .. against a column of large ones
    x[60, :] *= np.float32(2.0 ** 70)
    w[201, :] *= np.float32(2.0 ** -118)
    x[61, :] = 0.0
    got = _gpu_linear(rocm, lin, x, w, None).astype(np.float64)
    xf, wf = (np.where(np.isfinite(t), t, 0).astype(np.float64) for t in (x, w))
    mag = np.abs(xf) @ np.abs(wf).T
    with np.errstate(all="ignore"):
        exact = x.astype(np.float64) @ w.T.astype(np.float64)
    defined = mag < 3.0e38                               # elsewhere an fp32 sum may overflow on the way
    assert defined.mean() > 0.9 and np.isnan(exact[defined]).any() and np.isinf(exact[defined]).any()
    assert np.array_equal(np.isnan(got[defined]), np.isnan(exact[defined]))
    m = defined & np.isinf(exact)
    assert np.array_equal(got[m], exact[m])
    fine = defined & np.isfinite(exact)
    with np.errstate(all="ignore"):
        ok = np.abs(got - exact) <= (4.0 * np.sqrt(K) + 2.0) * EPS * mag + K * 2.0 ** -149   # a product below the floats' range is rounded to it
    assert ok[fine].all(), np.argwhere(fine & ~ok)[:5]
    assert fine[9, 100] and fine[50, 200] and fine[60, 201] and np.abs(exact[50, 200]) > 0 and got[61, 0] == 0


def test_fused_heads_see_the_plain_head(rocm, lin):  # noqa: F811
    """Greedy and sampling epilogues at shapes that take each tile: bit for bit the plain head's numbers."""
    from tests.test_gpu_linear import _fused_vs_unfused
    for M, N, K in [(48, 36000, 928), (100, 15000, 1088), (140, 33000, 352), (260, 66000, 96), (90, 3900, 4500)]:
        rng = np.random.default_rng(M)
        x = rng.standard_normal((M, K), dtype=np.float32)
        w = rng.standard_normal((N, K), dtype=np.float32) * np.float32(1.5 / np.sqrt(K))
        bias = np.float32(0.3) * rng.standard_normal(N, dtype=np.float32)
        hist = rng.integers(0, N, size=(M, 40)).astype(np.int32)
        _fused_vs_unfused(rocm, lin, x, w, bias, rocm.SamplerConfig(Temperature=0.7, TopK=50, TopP=0.9, RepetitionPenalty=1.15), hist)
        s = rocm.NewSampler(max_batch=M, max_vocab=N)
        layer = lin.Linear(K, N, rocm.DeviceBuffer.from_numpy(w), rocm.DeviceBuffer.from_numpy(bias))
        dx, logits, a, b = rocm.DeviceBuffer.from_numpy(x), rocm.DeviceBuffer(M * N * 4), rocm.DeviceBuffer(4 * M), rocm.DeviceBuffer(4 * M)
        layer.Forward(dx, (M, K), logits)
        s.Argmax(logits, M, N, a)
        lin.ForwardArgmax(s, layer, dx, (M, K), b)
        assert np.array_equal(a.to_numpy(np.int32, (M,)), b.to_numpy(np.int32, (M,))), (M, N, K)
        s.Close()


def test_rows_in_chunks(rocm, lin):  # noqa: F811
    """A left operand whose packed form exceeds the workspace is multiplied in chunks of rows."""
    M, K, N = 1900, 8192, 2600                             # (tests/test_gemm_plan.py holds it to more than one)
    rng = np.random.default_rng(3)
    x = rng.standard_normal((M, K), dtype=np.float32)
    w = rng.standard_normal((N, K), dtype=np.float32)
    got = _gpu_linear(rocm, lin, x, w, None)
    exact = x.astype(np.float64) @ w.T.astype(np.float64)
    assert np.all(np.abs(got - exact) <= _bound(x, w, None, K))


# (tests/test_gemm_plan.py holds these to more than one chunk: rows without slices of K, and with them)
@pytest.mark.parametrize("shape", [(2900, 2600, 4096), (700, 4096, 8192)])
def test_every_epilogue_in_chunks_of_rows(rocm, lin, shape):  # noqa: F811
    """The rows of every chunk, as the same rows alone give them: a chunk's offsets into the results, the greedy keys and the
    candidates' thresholds, counters and lists."""
    from tests.test_gpu_linear import _fused_vs_unfused
    M, N, K = shape
    rng = np.random.default_rng(M)
    x = rng.standard_normal((M, K), dtype=np.float32)
    w = rng.standard_normal((N, K), dtype=np.float32) * np.float32(1.5 / np.sqrt(K))
    bias = np.float32(0.3) * rng.standard_normal(N, dtype=np.float32)
    layer = lin.Linear(K, N, rocm.DeviceBuffer.from_numpy(w), rocm.DeviceBuffer.from_numpy(bias))
    dx, logits = rocm.DeviceBuffer.from_numpy(x), rocm.DeviceBuffer(M * N * 4)
    layer.Forward(dx, (M, K), logits)
    got = logits.to_numpy(np.float32, (M, N))
    rows = np.unique(np.concatenate([np.arange(0, M, 97), [255, 256, 257, 511, 512, 1023, 1024, 1535, 1536, M - 1]]))
    rows = rows[rows < M]
    exact = x[rows].astype(np.float64) @ w.T.astype(np.float64) + bias[None, :]
    assert np.all(np.abs(got[rows] - exact) <= _bound(x[rows], w, bias, K))
    s, a, b = rocm.NewSampler(max_batch=M, max_vocab=N), rocm.DeviceBuffer(4 * M), rocm.DeviceBuffer(4 * M)
    s.Argmax(logits, M, N, a)
    lin.ForwardArgmax(s, layer, dx, (M, K), b)
    assert np.array_equal(a.to_numpy(np.int32, (M,)), b.to_numpy(np.int32, (M,)))
    s.Close()
    hist = rng.integers(0, N, size=(M, 8)).astype(np.int32)
    _fused_vs_unfused(rocm, lin, x, w, bias, rocm.SamplerConfig(Temperature=0.7, TopK=20, TopP=0.9, RepetitionPenalty=1.15), hist)
