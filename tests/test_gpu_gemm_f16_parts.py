"""Large products in two fp16 parts (born_amd/csrc/gemm_split.hip, K from 256 on): operands that their scales or their range do not fit, and rows and
columns for which two parts are not enough and which have to be whole.

Tolerance: that of tests/test_gpu_linear.py, (4 sqrt(K) + 2) 2^-24 (sum |a| |b|), result by result.  Two parts hold a value to 2^-23 of it and leave
2^-22 of a product out at most, 8 of the bound's more than 66 units together; values too small for that are looked after apart.
"""
import numpy as np
import pytest

from tests.test_gpu_linear import _bound, _gpu_linear, _gpu_matmul, lin, rocm  # noqa: F401  (fixtures)

pytestmark = pytest.mark.gpu

# a tile of each height; K at the first of two parts, at one past a group, and odd; ragged M and N
SHAPES = [(17, 45000, 2048), (32, 24500, 2049), (48, 130000, 256), (100, 15011, 1057), (130, 40004, 300), (270, 16000, 352), (64, 6100, 4096)]


def _operands(kind, rng, M, N, K):
    x, w = rng.standard_normal((M, K), dtype=np.float32), rng.standard_normal((N, K), dtype=np.float32)
    if kind == "few terms of every magnitude":                # a result is one or two products, down to 2^-60 of the largest
        keep = rng.integers(0, K, (M, 2))
        y = np.zeros_like(x)
        y[np.arange(M)[:, None], keep] = x[np.arange(M)[:, None], keep]
        return y, np.ldexp(w, rng.integers(-60, 1, (N, K))).astype(np.float32)
    if kind == "rows of a wide range":
        return np.ldexp(x, rng.integers(-70, 1, (M, K))).astype(np.float32), w
    if kind == "one huge factor that meets zeros":
        x[:, K // 2] = np.float32(2.0 ** 100)
        w[:, K // 2] = 0
        return x, w
    if kind == "columns that begin with zeros":               # the scale comes from other columns, or there is none
        w[::3, :200] = 0
        w[N // 2: N // 2 + 100, :200] = 0
        w[::9] = 0
        w[1::64] *= np.float32(2.0 ** -40)
        x[1::5] = 0
        return x, w
    if kind == "few values in a column":                      # now and then small ones first
        return x, np.where(rng.random((N, K), dtype=np.float32) < 0.03, np.ldexp(w, rng.integers(-12, 1, (N, K))), 0).astype(np.float32)
    if kind == "equal rows":                                  # a small result in one is small in all, some over values that are cut
        x[:] = x[0]
        w[:, 5::64] *= np.float32(2.0 ** -24)
        return x, w
    if kind == "signs and zeros":                             # results of zero by the score
        return rng.integers(-1, 2, (M, K)).astype(np.float32), rng.integers(-1, 2, (N, K)).astype(np.float32) * np.float32(0.37)
    if kind == "late large values":                          # the tiles that begin before them are done again
        w[:, K // 2:] *= 1000
        return x, w
    if kind == "heavy tails":
        return x, w / np.maximum(np.abs(rng.standard_normal((N, K), dtype=np.float32)), np.float32(1e-6))
    if kind == "columns that outgrow their scale":
        w[::1000, K - 3:] *= np.float32(2.0 ** 30)
        w[5::1000, K - 3:] *= np.float32(2.0 ** -30)
        return x, w
    x *= np.ldexp(np.float32(1), rng.integers(-60, 61, (M, 1))).astype(np.float32)   # every row and column in units of its own
    w *= np.ldexp(np.float32(1), rng.integers(-60, 61, (N, 1))).astype(np.float32)
    return x, w


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("kind", ["few terms of every magnitude", "rows of a wide range", "one huge factor that meets zeros",
                                  "columns that begin with zeros", "few values in a column", "equal rows", "signs and zeros", "late large values", "heavy tails", "columns that outgrow their scale", "units"])
def test_every_result_keeps_its_precision(rocm, lin, kind, shape):  # noqa: F811
    M, N, K = shape
    rng = np.random.default_rng(K)
    x, w = _operands(kind, rng, M, N, K)
    some = np.unique(np.concatenate([rng.choice(N, 1500, replace=False), [0, N - 1, *range(0, N, 1000), *range(5, N, 1000)]]))
    got = _gpu_linear(rocm, lin, x, w, None)[:, some] if N % 2 else _gpu_matmul(rocm, lin, x, np.ascontiguousarray(w.T))[:, some]
    exact = x.astype(np.float64) @ w[some].T.astype(np.float64)
    err = np.abs(got - exact) - 2.0 ** -140 * K             # (products below the floats' range)
    bound = _bound(x, w[some], None, K)
    assert np.all(err <= bound), (kind, shape, np.argwhere(err > bound)[:3], (err / np.maximum(bound, 1e-300)).max())


def test_values_cut_under_columns_far_above_their_scale(rocm, lin):  # noqa: F811
    """A row of one large value that meets zeros and many equal ones 2^-32 of it, whose parts are cut (all alike, so that nothing averages out), against
    columns whose later values are 256 times those their scale is made from: what is lost shows in results of any size, so they are summed again.
    Sixteen units: sums of fp32 products in pieces of 512 are off by the walk of 128 roundings, three or four."""
    M, N, K = 40, 33000, 4096                                # (K in one piece: a slice's partial sums are smaller)
    rng = np.random.default_rng(3)
    x = rng.standard_normal((M, K), dtype=np.float32)
    w = rng.random((N, K), dtype=np.float32) * np.float32(0.09) + np.float32(1.9)
    w[:, 64:] *= 256
    w[:, 4000] = 0
    rows, some = np.arange(1, M, 7), rng.choice(N, 1000, replace=False)
    x[rows] = np.float32(1.007) * np.float32(2.0 ** -32)
    x[rows, 4000] = 1
    got = _gpu_linear(rocm, lin, x, w, None)[np.ix_(rows, some)]
    exact = x[rows].astype(np.float64) @ w[some].T.astype(np.float64)
    assert (np.abs(got - exact) / exact).max() <= 16 * 2.0 ** -24


# every tile, by 128-bit loads and value by value; ragged M, N and K, and K in slices (64 x 6100, 128 x 6000)
WHOLE_SHAPES = [(20, 45001, 2048), (48, 130000, 257), (100, 15011, 1057), (130, 40004, 300), (270, 16000, 352), (64, 6100, 4096),
                (128, 6000, 4096), (128, 6001, 4099), (300, 40001, 517), (512, 20001, 513)]


def _both_forms(rocm, lin, x, w):
    yield _gpu_linear(rocm, lin, x, w, None)
    yield _gpu_matmul(rocm, lin, x, np.ascontiguousarray(w.T))


@pytest.mark.parametrize("shape", WHOLE_SHAPES)
def test_rows_and_columns_that_select_are_exact(rocm, lin, shape):  # noqa: F811
    """One power of two in a row: a row of the weights, bit for bit; one in a column: the activations."""
    M, N, K = shape
    rng = np.random.default_rng(K)
    x, w = rng.standard_normal((M, K), dtype=np.float32), rng.standard_normal((N, K), dtype=np.float32)
    rows, at = np.arange(1, M, 9), rng.integers(0, K, len(range(1, M, 9)))
    x[rows] = 0
    x[rows, at] = np.ldexp(np.float32(1), rng.integers(-3, 4, len(rows))).astype(np.float32) * rng.choice(np.array([-1, 1], np.float32), len(rows))
    for got in _both_forms(rocm, lin, x, w):
        assert np.array_equal(got[rows], w[:, at].T * x[rows, at][:, None])
    x = rng.standard_normal((M, K), dtype=np.float32)
    cols, of = rng.choice(N, 700, replace=False), rng.integers(0, K, 700)
    w[cols] = 0
    w[cols, of] = np.float32(0.25)
    for got in _both_forms(rocm, lin, x, w):
        assert np.array_equal(got[:, cols], x[:, of] * np.float32(0.25))


@pytest.mark.parametrize("shape", WHOLE_SHAPES)
def test_a_product_of_two_whole_values_is_rounded_once(rocm, lin, shape):  # noqa: F811
    """Rows of one term: six of nine products of parts, their small ones in a sum of their own that is off by 2^-11 of a unit."""
    M, N, K = shape
    rng = np.random.default_rng(K + 1)
    x, w = np.zeros((M, K), np.float32), rng.standard_normal((N, K), dtype=np.float32)
    at = rng.integers(0, K, M)
    x[np.arange(M), at] = rng.standard_normal(M, dtype=np.float32)
    for got in _both_forms(rocm, lin, x, w):
        exact = x[np.arange(M), at].astype(np.float64)[:, None] * w[:, at].T.astype(np.float64)
        assert np.all(np.abs(got - exact) <= 2.0 ** -24 * (1 + 2.0 ** -8) * np.abs(exact))


@pytest.mark.parametrize("shape", WHOLE_SHAPES)
def test_whole_numbers_are_exact(rocm, lin, shape):  # noqa: F811
    """Sums below 2^24 of products whose factors both need their second part, and of factors of 22 bits."""
    M, N, K = shape
    rng = np.random.default_rng(K + 2)
    x, w = rng.integers(-20, 21, (M, K)).astype(np.float32), rng.integers(-20, 21, (N, K)).astype(np.float32)
    x[:, K // 2], w[:, K // 2] = rng.integers(2049, 2600, M), rng.integers(2049, 2600, N)
    x[:, 7], w[:, 7] = rng.integers(2 ** 21, 2 ** 22, M), rng.integers(-1, 2, N)
    assert (np.abs(x).astype(np.float64) @ np.abs(w[:2000]).T.astype(np.float64)).max() < 2.0 ** 24
    want = (x.astype(np.float64) @ w.T.astype(np.float64)).astype(np.float32)
    for got in _both_forms(rocm, lin, x, w):
        assert np.array_equal(got, want)


# what two fp16 parts lose most of: the product of the second parts; that, and a unit of either factor
SIGNIFICANDS = [1 + 2.0 ** -11, 1 + 2.0 ** -11 - 3 * 2.0 ** -23]


@pytest.mark.parametrize("K", [256, 1000, 4096])
@pytest.mark.parametrize("family", ["equal", "signed", "powers", "4 terms", "12 terms"])
@pytest.mark.parametrize("value", SIGNIFICANDS)
def test_error_is_that_of_whole_operands(rocm, lin, family, value, K):  # noqa: F811
    """The 2-norm of the error against fp64, beside that of the same rows 16 at a time, which the fp32 tiles multiply.  What two parts lose is
    up to 8 units of 2^-24 here; two roundings to a group of 32 are a walk of sqrt(K / 16) / 3 units (rounded the same way by equal terms: one and a half of
    it), and the result is rounded once."""
    M, N = 64, int(3.1e9 / (2 * 64 * K))
    rng = np.random.default_rng(K)
    sign = lambda rows: rng.choice(np.array([-1, 1], np.float32), (rows, K))  # noqa: E731
    x, w = np.full((M, K), np.float32(value)), np.full((N, K), np.float32(value))
    if family == "signed":
        x, w = x * sign(M), w * sign(N)
    elif family == "powers":                                 # one significand, every value a power of two of its own
        x, w = np.ldexp(x, rng.integers(-3, 4, (M, K))).astype(np.float32), np.ldexp(w, rng.integers(-3, 4, (N, K))).astype(np.float32)
    elif family != "equal":
        keep = np.argsort(rng.random((M, K)), axis=1)[:, int(family.split()[0]):]
        np.put_along_axis(x, keep, np.float32(0), 1)
        w = rng.standard_normal((N, K), dtype=np.float32)
    some = rng.choice(N, min(N, 2000), replace=False)
    layer, dx = lin.Linear(K, N, rocm.DeviceBuffer.from_numpy(w), None), rocm.DeviceBuffer.from_numpy(x)
    one, two = rocm.DeviceBuffer(M * N * 4), rocm.DeviceBuffer(M * N * 4)
    layer.Forward(dx, (M, K), one)
    for r in range(0, M, 16):
        layer.Forward(dx.ptr + 4 * r * K, (16, K), two.ptr + 4 * r * N)
    exact = x.astype(np.float64) @ w[some].T.astype(np.float64)
    split, tiles = (np.sqrt(np.mean((b.to_numpy(np.float32, (M, N))[:, some] - exact) ** 2) / np.mean(exact ** 2)) for b in (one, two))
    print(f"{family} {value} {K}: {split * 2 ** 24:.3f} {tiles * 2 ** 24:.3f} units")
    assert split <= max(1.03 * tiles, (1 + np.sqrt(K / 16) / 2) * 2.0 ** -24), (split, tiles)


@pytest.mark.parametrize("shape", [(48, 36000, 928), (140, 33000, 352), (300, 40001, 517), (260, 66000, 300)])
def test_fused_heads_see_the_plain_head_s_whole_rows(rocm, lin, shape):  # noqa: F811
    """Batches of which a tile is whole and others may not be: bit for bit the plain head's numbers."""
    from tests.test_gpu_linear import _fused_vs_unfused
    M, N, K = shape
    rng = np.random.default_rng(M)
    x = rng.standard_normal((M, K), dtype=np.float32)
    x[3] = 0
    x[3, 5], x[M - 1] = 2, np.round(1000 * x[M - 1])
    w = rng.standard_normal((N, K), dtype=np.float32) * np.float32(1.5 / np.sqrt(K))
    bias = np.float32(0.3) * rng.standard_normal(N, dtype=np.float32)
    x[M - 1] /= 1024
    hist = rng.integers(0, N, size=(M, 40)).astype(np.int32)
    _fused_vs_unfused(rocm, lin, x, w, bias, rocm.SamplerConfig(Temperature=0.7, TopK=50, TopP=0.9, RepetitionPenalty=1.15), hist)
    s = rocm.NewSampler(max_batch=M, max_vocab=N)
    layer = lin.Linear(K, N, rocm.DeviceBuffer.from_numpy(w), rocm.DeviceBuffer.from_numpy(bias))
    dx, logits, a, b = rocm.DeviceBuffer.from_numpy(x), rocm.DeviceBuffer(M * N * 4), rocm.DeviceBuffer(4 * M), rocm.DeviceBuffer(4 * M)
    layer.Forward(dx, (M, K), logits)
    s.Argmax(logits, M, N, a)
    lin.ForwardArgmax(s, layer, dx, (M, K), b)
    assert np.array_equal(a.to_numpy(np.int32, (M,)), b.to_numpy(np.int32, (M,)))
    s.Close()


@pytest.mark.parametrize("shape", [(64, 24000, 1024), (100, 15011, 1057), (128, 12000, 1024), (300, 16000, 1024)])
def test_sums_of_nothing_but_tiny_products(rocm, lin, shape):  # noqa: F811
    """Values far below their row's and column's largest, none of which is cut, where those largest meet zeros: the accumulators do not hold such sums."""
    M, N, K = shape
    rng = np.random.default_rng(K)
    x, w = rng.standard_normal((M, K), dtype=np.float32), np.zeros((N, K), np.float32)
    rows = np.arange(2, M, 3)
    sized = lambda *s: (1 + rng.random(s, dtype=np.float32)) * rng.choice(np.array([-1, 1], np.float32), s)  # noqa: E731
    w[:, ::16] = 1
    w[:, [41, 700]] = np.float32(2.0 ** -18) * sized(N, 2)
    x[rows] = 0
    x[rows, 300] = 1
    x[np.ix_(rows, [41, 700])] = np.float32(2.0 ** -25) * sized(len(rows), 2)
    for got in _both_forms(rocm, lin, x, w):
        exact = x[rows].astype(np.float64) @ w.T.astype(np.float64)
        err = np.abs(got[rows] - exact) / _bound(x[rows], w, None, K)
        assert err.max() <= 1, err.max()


@pytest.mark.parametrize("shape", [(64, 24000, 1024), (100, 15011, 1057), (128, 12000, 1024), (300, 16000, 1024)])
def test_columns_that_outgrow_their_scale_lose_nothing(rocm, lin, shape):  # noqa: F811
    """The 2-norm of the error of columns whose second half is 1000 times their first, beside that of the same columns reversed, which begin with their
    largest: both are sums of the same products in groups of 32, one and a half walks of their roundings at most."""
    M, N, K = shape
    rng = np.random.default_rng(K)
    x, w = rng.standard_normal((M, K), dtype=np.float32), rng.standard_normal((N, K), dtype=np.float32)
    w[:, K // 2:] *= 1000
    some = rng.choice(N, 2000, replace=False)
    exact = x.astype(np.float64) @ w[some].T.astype(np.float64)
    size = np.sqrt(np.mean(exact ** 2))
    rms = lambda got: np.sqrt(np.mean((got[:, some] - exact) ** 2)) / size  # noqa: E731
    late, early = rms(_gpu_linear(rocm, lin, x, w, None)), rms(_gpu_linear(rocm, lin, x[:, ::-1].copy(), w[:, ::-1].copy(), None))
    print(f"{shape}: {late * 2 ** 24:.2f} and {early * 2 ** 24:.2f} units")
    assert late <= 1.3 * early and late <= (1 + np.sqrt(K / 16) / 2) * 2.0 ** -24, (late, early)
