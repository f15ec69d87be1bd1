"""Large products in two fp16 parts (born_amd/csrc/gemm_split.hip, K from 256 on): operands that their scales or their range do not fit.

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
    if kind == "columns that outgrow their scale":
        w[::1000, K - 3:] *= np.float32(2.0 ** 30)
        w[5::1000, K - 3:] *= np.float32(2.0 ** -30)
        return x, w
    x *= np.ldexp(np.float32(1), rng.integers(-60, 61, (M, 1))).astype(np.float32)   # every row and column in units of its own
    w *= np.ldexp(np.float32(1), rng.integers(-60, 61, (N, 1))).astype(np.float32)
    return x, w


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("kind", ["few terms of every magnitude", "rows of a wide range", "one huge factor that meets zeros",
                                  "columns that begin with zeros", "columns that outgrow their scale", "units"])
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
