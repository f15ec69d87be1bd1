"""How a row's logits are read, by its start, pitch and length: aligned rows, rows of any start by 128-bit loads, short ones one logit
at a time.  Every form at the lengths where the kernels change from one to the other, against the oracle's fixed-point layer, bit for
bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# around 1536 (three sweeps, verification), 3584 and 8192 (top-k with 512 and 1024 threads), 4096 (general kernel)
LENGTHS = [1000, 1535, 1537, 3583, 3585, 4095, 4097, 8191, 8193]
FORMS = [(0, 0), (1, 0), (0, 3), (2, 1)]                    # (floats in front of the first row, floats between rows beyond a multiple of 4)


@pytest.fixture(scope="module")
def rocm():
    from born_amd import sampler as S
    assert S.DeviceCount() >= 1, "no HIP device visible"
    return S


def _laid_out(rocm, x, before, pitch):
    """The rows at `pitch` floats, `before` floats into a buffer whose other values would win every draw."""
    B, V = x.shape
    flat = np.full(before + B * pitch, 1e6, np.float32)
    rows = flat[before:].reshape(B, pitch)
    rows[:, :V] = x
    buf = rocm.DeviceBuffer.from_numpy(flat)
    return buf, buf.ptr + 4 * before


@pytest.mark.parametrize("path", [0, 1, 2])                 # 1: the general kernel; 2: 512 threads to a row
@pytest.mark.parametrize("k,p,T", [(40, 0.95, 0.8), (200, 1.0, 1.0), (0, 0.95, 0.8), (0, 1.0, 1.0)])
@pytest.mark.parametrize("before,over", FORMS)
def test_sampling(oracle, rocm, before, over, k, p, T, path):
    for V in LENGTHS:
        rng = np.random.default_rng(V)
        B, pitch = 5, (V + 3) // 4 * 4 + over
        x = rng.standard_normal((B, V)).astype(np.float32)
        x[1::2, V - 3:] += np.float32(6)
        u, hist = rng.random(B).astype(np.float32), np.tile(np.array([[V - 1, 0, V - 3]], np.int32), (B, 1))
        buf, at = _laid_out(rocm, x, before, pitch)
        d_u, d_h, tok, pr = rocm.DeviceBuffer.from_numpy(u), rocm.DeviceBuffer.from_numpy(hist), rocm.DeviceBuffer(4 * B), rocm.DeviceBuffer(4 * B)
        s = rocm.NewSampler(rocm.SamplerConfig(Temperature=T, TopK=k, TopP=p, RepetitionPenalty=1.2), max_batch=B, max_vocab=V)
        s.SetPath(path)
        s.Sample(at, B, V, d_h, None, d_u, tok, pr, row_stride=pitch, hist_stride=3)
        s.Status()
        s.Close()
        want = oracle.sample(x, u, T, k, p, 1.2, hist, mode=oracle.MODE_FIXED)
        assert np.array_equal(tok.to_numpy(np.int32, (B,)), want["tokens"]), V
        assert np.array_equal(pr.to_numpy(np.uint32, (B,)), want["probs"].view(np.uint32)), V


@pytest.mark.parametrize("T", [1.0, 0.8])
@pytest.mark.parametrize("V", [1000, 1535, 1537, 3073, 32767, 32768])
def test_verification(oracle, rocm, V, T):
    rng = np.random.default_rng(V)
    B, G = 3, 2
    t = rng.standard_normal((B, G + 1, V)).astype(np.float32)
    d = (t[:, :G] + rng.standard_normal((B, G, V))).astype(np.float32)
    t[::2, :, V - 2:] += np.float32(4)
    tok = rng.integers(0, V, (B, G)).astype(np.int32)
    tok[1] = d[1].argmax(-1)
    ua, ur = rng.random((B, G)).astype(np.float32), rng.random(B).astype(np.float32)
    ua[1] = 0                                              # accepted whole: the bonus row is drawn from
    want = oracle.spec_verify(t[:, :G], d, tok, ua, ur, temperature=T, mode=oracle.MODE_FIXED, bonus=t[:, G])
    dev = [rocm.DeviceBuffer.from_numpy(a) for a in (tok, ua, ur)]
    for before, over in FORMS:                             # (a sequence's rows follow each other: a pitch per sequence)
        pt, pd = (G + 1) * V + over, G * V + over
        bt, at = _laid_out(rocm, t.reshape(B, -1), before, pt)
        bd, ad = _laid_out(rocm, d.reshape(B, -1), before, pd)
        s = rocm.NewSampler(rocm.SamplerConfig(Temperature=T), max_batch=B, max_vocab=V)
        n, nxt = rocm.DeviceBuffer(4 * B), rocm.DeviceBuffer(4 * B)
        s.VerifyBonus(at, pt, ad, pd, at + 4 * G * V, pt, B, G, V, *dev, n, nxt)
        s.Status()
        s.Close()
        assert np.array_equal(n.to_numpy(np.int32, (B,)), want["n_accepted"]), (before, over)
        assert np.array_equal(nxt.to_numpy(np.int32, (B,)), want["next_token"]), (before, over)


def test_rows_with_temperatures_at_the_ends_of_the_reciprocal(oracle, rocm):
    """A row's own temperature is divided by through its reciprocal from 2^-20 to 2^20; the logits span a few temperatures."""
    f = np.float32
    ends = [f(2.0 ** -20), np.nextafter(f(2.0 ** -20), f(0)), f(2.0 ** 20), np.nextafter(f(2.0 ** 20), f(np.inf)), f(1), f(0.7), f(1.9999999)]
    Ts = np.array(ends * 2, np.float32)
    for V, path in ((1001, 0), (9001, 0), (9001, 2)):
        rng = np.random.default_rng(V)
        B = len(Ts)
        x = (rng.standard_normal((B, V)) * 2 * Ts[:, None]).astype(np.float32)
        x[:, 5], x[:, 6], x[:, 7] = 0, -np.inf, np.nan
        u, ps = rng.random(B).astype(np.float32), np.where(np.arange(B) < len(ends), f(0.9), f(1)).astype(np.float32)
        s = rocm.NewSampler(rocm.SamplerConfig(), max_batch=B, max_vocab=V)
        s.SetPath(path)
        dev = [rocm.DeviceBuffer.from_numpy(a) for a in (x, u, Ts, ps)]
        tok, pr = rocm.DeviceBuffer(4 * B), rocm.DeviceBuffer(4 * B)
        s.SampleRows(dev[0], B, V, None, None, dev[1], dev[2], None, dev[3], None, tok, pr)
        s.Status()
        s.Close()
        for b in range(B):
            want = oracle.sample(x[b:b + 1], u[b:b + 1], Ts[b], 0, ps[b], 1.0, None, mode=oracle.MODE_FIXED)
            assert tok.to_numpy(np.int32, (B,))[b] == want["tokens"][0], (V, b)
            assert pr.to_numpy(np.uint32, (B,))[b] == want["probs"].view(np.uint32)[0], (V, b)
