"""The verification's masses summed in fp64: lengths around where the sum's room and the way of reading change, rows of equal logits (the
fullest sums), rows whose masses mostly truncate to nothing, and uniforms at the very ratio of the two models' masses, which a sum off by 2^-22 moves
to the other side.  Against the oracle's fixed-point layer."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1.0, 0.7])
@pytest.mark.parametrize("V", [4, 508, 511, 512, 1024, 1536, 1540, 2047, 2048, 2052, 4095, 4096, 4100, 16384, 32764, 32767, 32768, 32769, 36863, 65535, 65536, 131071])
def test_verification(oracle, V, T):
    from born_amd import sampler as S
    rng = np.random.default_rng(V)
    B, G = 4, 2
    t = np.full((B, G + 1, V), 3.0, np.float32)                       # (a maximum of 0 would be no usual row)
    d = t[:, :G].copy()
    d[1] += rng.standard_normal((G, V)).astype(np.float32)
    t[2] -= (40 * rng.random((G + 1, V))).astype(np.float32)         # down to masses far below 2^-S
    t[3], d[3] = 2 * rng.standard_normal((G + 1, V)), 2 * rng.standard_normal((G, V))
    tok = rng.integers(0, V, (B, G)).astype(np.int32)

    def p(x, i):
        e = np.exp((x.astype(np.float64) - x.max()) / T)
        return e[i] / e.sum()

    ratio = np.array([[p(t[b, g], tok[b, g]) / p(d[b, g], tok[b, g]) for g in range(G)] for b in range(B)])
    for off in (-1.0, 1.0):                                           # 2^-22 of the ratio to either side
        ua = np.clip(ratio * (1 + off * 2.0 ** -22), 0, 1 - 2.0 ** -24).astype(np.float32)
        ur = rng.random(B).astype(np.float32)
        s = S.NewSampler(S.SamplerConfig(Temperature=T), max_batch=B, max_vocab=V)
        got = S.verify_host(s, t, d, tok, ua, ur, bonus=True)
        s.Status()
        s.Close()
        want = oracle.spec_verify(np.ascontiguousarray(t[:, :G]), d, tok, ua, ur, temperature=T, mode=oracle.MODE_FIXED, bonus=np.ascontiguousarray(t[:, G]))
        assert np.array_equal(got["n_accepted"], want["n_accepted"]) and np.array_equal(got["next_token"], want["next_token"]), off


@pytest.mark.parametrize("V", [64, 256, 2047, 2048, 2049, 4096, 8191, 8192, 8193, 16383, 16384, 16385, 32767, 32768, 32769, 65535, 65536, 100001])
def test_softmax(oracle, V):
    """Rows of equal logits (each sum as full as it gets), of masses that truncate, with NaNs, infinities of both signs and zeros: the masses' sum is the
    oracle's to the bit in softmax, and log-softmax is the specified expression of it within the rounding of its logarithm."""
    from born_amd import sampler as S
    rng = np.random.default_rng(V)
    x = np.zeros((7, V), np.float32)
    x[1] = -3.0
    x[2] = -(60 * rng.random(V)).astype(np.float32)
    x[3], x[4] = 3 * rng.standard_normal(V), 3 * rng.standard_normal(V)
    x[3, ::5], x[3, 1::7], x[3, 2] = np.nan, -np.inf, -3e38
    x[4, V // 2] = np.inf
    x[5] = -np.inf
    x[6, 1:] = -100 - rng.random(V - 1)
    s = S.NewSampler(max_batch=7, max_vocab=V)
    d, o = S.DeviceBuffer.from_numpy(x), S.DeviceBuffer(x.nbytes)
    z = np.minimum(np.where(np.isnan(x), -np.inf, x), np.float32(3.402823466e38)).astype(np.float32)
    m = z.max(1)
    with np.errstate(invalid="ignore", over="ignore"):
        dist = np.where(z == m[:, None], np.float32(0), (m[:, None] - z).astype(np.float32)).astype(np.float32)
    e = oracle.expneg(dist).astype(np.float64)
    S2 = 62 - int(V).bit_length()
    Z = np.array([float(sum(int(v) for v in np.trunc(row * 2.0 ** S2))) for row in e]) * 2.0 ** -S2
    s.Softmax(d, 7, V, o)
    assert np.array_equal(o.to_numpy(np.uint32, x.shape), (e / Z[:, None]).astype(np.float32).view(np.uint32))
    s.Softmax(d, 7, V, o, log=True)
    got = o.to_numpy(np.float32, x.shape)
    with np.errstate(invalid="ignore"):
        want = ((z.astype(np.float64) - m[:, None].astype(np.float64)) - np.log(Z)[:, None]).astype(np.float32)
    same = (got == want) | (np.abs(got - want) <= 2.0 ** -23 * np.abs(want)) | (np.isnan(got) & np.isnan(want))   # (the logarithm's last place)
    assert same.all()
    s.Close()
