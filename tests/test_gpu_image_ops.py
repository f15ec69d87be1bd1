"""Operations on images at the edges of their kernels: convolutions without padding by one, two and four channels a lane, planes of one position and of
whole blocks, strides, channel counts around the pairs of the loop; a bias per channel with the last dimension a multiple of four or not, either
operand broadcast; pools of the unrolled sizes and others.  Bit for bit against the oracle's restatement of the reference."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,C,H,W,CO,K,stride", [
    (1, 1, 5, 5, 1, 5, 1), (1, 1, 3, 3, 3, 3, 1), (3, 2, 7, 9, 5, 5, 1), (2, 3, 8, 8, 6, 3, 2), (5, 5, 12, 11, 7, 5, 3), (9, 4, 20, 20, 33, 5, 1), (40, 2, 20, 20, 21, 5, 1),
    (64, 1, 28, 28, 32, 5, 1), (16, 3, 34, 34, 50, 3, 1), (17, 6, 30, 30, 11, 3, 1), (64, 32, 12, 12, 64, 5, 1), (270, 2, 32, 32, 1, 5, 1), (720, 1, 32, 32, 1, 3, 1),
    (360, 1, 32, 32, 2, 5, 1), (320, 2, 32, 32, 2, 3, 1), (240, 2, 32, 32, 3, 5, 1)])
def test_convolution(oracle, N, C, H, W, CO, K, stride):
    from born_amd import backend as BK
    rng = np.random.default_rng(N * 1000 + CO)
    x, k = rng.standard_normal((N, C, H, W)).astype(np.float32), rng.standard_normal((CO, C, K, K)).astype(np.float32)
    x[0, 0, 0, 0], x[-1, -1, -1, -1] = np.inf, -0.0
    got = BK.New().Conv2D(BK.DeviceTensor.from_numpy(x), BK.DeviceTensor.from_numpy(k), stride, 0).numpy()
    want = oracle.conv2d_ref(x, k, stride, 0)
    assert got.shape == want.shape
    assert ((got.view(np.uint32) == want.view(np.uint32)) | (np.isnan(got) & np.isnan(want))).all()


@pytest.mark.parametrize("a,b", [((3, 5, 6, 6), (1, 5, 1, 1)), ((3, 5, 5, 5), (1, 5, 1, 1)), ((1, 7, 1, 1), (2, 7, 4, 8)), ((4, 1, 9), (1, 3, 1)), ((2, 3, 4), (2, 1, 4)),
                                 ((2, 3, 5), (2, 1, 5)), ((3, 1, 8), (1, 4, 8)), ((64, 32, 24, 24), (1, 32, 1, 1)), ((2, 1, 3, 4), (1, 5, 1, 4))])
def test_broadcast_of_three_dimensions(oracle, a, b):
    from born_amd import backend as BK
    rng = np.random.default_rng(len(a) + sum(a))
    x, y = rng.standard_normal(a).astype(np.float32), (rng.standard_normal(b) + 3).astype(np.float32)
    be = BK.New()
    for op, f in (("add", be.Add), ("sub", be.Sub), ("mul", be.Mul), ("div", be.Div)):
        got, want = f(BK.DeviceTensor.from_numpy(x), BK.DeviceTensor.from_numpy(y)).numpy(), oracle.binary_ref(op, x, y)
        assert got.shape == want.shape and np.array_equal(got.view(np.uint32), want.view(np.uint32)), op


@pytest.mark.parametrize("shape,size,stride", [((2, 3, 2, 2), 2, 2), ((64, 32, 24, 24), 2, 2), ((3, 5, 9, 11), 3, 2), ((3, 5, 9, 11), 2, 3), ((1, 2, 7, 7), 5, 1), ((2, 2, 6, 6), 1, 1)])
def test_pool(oracle, shape, size, stride):
    from born_amd import backend as BK
    x = np.random.default_rng(size).standard_normal(shape).astype(np.float32)
    x[0, 0, 0, 0], x[0, 1, :2, :2] = np.nan, -np.inf
    got = BK.New().MaxPool2D(BK.DeviceTensor.from_numpy(x), size, stride).numpy()
    want = oracle.maxpool2d_ref(x, size, stride)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
