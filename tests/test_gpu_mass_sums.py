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
