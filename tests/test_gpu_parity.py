"""GPU parity tests: the HIP path (through the C ABI) against the CPU oracle on the same seeded inputs.

Bars (docs/SAMPLING_SPEC.md):
  * against the fixed-point layer of the oracle: token ids, nucleus sizes, accept counts — bit-exact,
    every row; probabilities bit-exact as fp32;
  * against the fp64 truth layer: token ids equal except on rows the truth layer flags as drawn within
    1e-6 of a CDF step (counted, bounded); probabilities within 1e-5 relative.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rocm():
    from born_amd import sampler as S
    assert S.DeviceCount() >= 1, "no HIP device visible"
    return S


def _run(rocm, x, u, T=1.0, k=0, p=1.0, rep=1.0, hist=None, hist_len=None, nuc=0, path=0, max_vocab=None, min_p=0.0,
         freq=0.0, pres=0.0):
    B, V = x.shape
    s = rocm.NewSampler(rocm.SamplerConfig(Temperature=T, TopK=k, TopP=p, RepetitionPenalty=rep, MinP=min_p,
                                           FrequencyPenalty=freq, PresencePenalty=pres), max_batch=B, max_vocab=max_vocab or V)
    s.SetPath(path)
    out = rocm.sample_host(s, x, u, hist, hist_len, nucleus_cap=nuc)
    out["counters"] = s.Counters()
    s.Status()
    s.Close()
    return out


def _check_against_oracle(oracle, rocm, x, u, T=1.0, k=0, p=1.0, rep=1.0, hist=None, hist_len=None, nuc=0, path=0,
                          max_near_frac=1.0, min_p=0.0, freq=0.0, pres=0.0):
    got = _run(rocm, x, u, T, k, p, rep, hist, hist_len, nuc, path, min_p=min_p, freq=freq, pres=pres)
    fx = oracle.sample(x, u, T, k, p, rep, hist, hist_len, mode=oracle.MODE_FIXED, nuc_cap=nuc, min_p=min_p, freq=freq, pres=pres)
    tr = oracle.sample(x, u, T, k, p, rep, hist, hist_len, mode=oracle.MODE_TRUTH, nuc_cap=nuc, min_p=min_p, freq=freq, pres=pres)
    bad = np.nonzero(got["tokens"] != fx["tokens"])[0]
    assert bad.size == 0, f"token mismatch vs fixed-point oracle at rows {bad[:8]}: {got['tokens'][bad[:8]]} vs {fx['tokens'][bad[:8]]}"
    assert np.array_equal(got["probs"].view(np.uint32), fx["probs"].view(np.uint32)), "probabilities differ from the fixed-point oracle"
    diff = got["tokens"] != tr["tokens"]
    assert not (diff & ~tr["near"]).any(), "token differs from the fp64 truth on a row not flagged near a CDF step"
    assert tr["near"].mean() <= max_near_frac
    # (a row whose top-p / min-p cut lies within the tolerance of an element boundary may keep one element more or fewer
    # in the truth layer than in the fixed-point layer: same token, another normaliser; the truth layer flags such rows)
    same = ~diff & ~tr["near_cut"]
    assert np.allclose(got["probs"][same], tr["probs"][same], rtol=1e-5, atol=0), "probability off by more than 1e-5 relative"
    if nuc:
        assert np.array_equal(got["n_nucleus"], fx["n_nucleus"])
        assert np.array_equal(got["nuc_ids"], fx["nuc_ids"])
        assert np.array_equal(got["nuc_probs"].view(np.uint32), fx["nuc_probs"].view(np.uint32))
        ok = ~tr["near_cut"]
        assert np.array_equal(got["n_nucleus"][ok], tr["n_nucleus"][ok])
        m = (tr["nuc_ids"][ok] >= 0) & (tr["nuc_ids"][ok] == got["nuc_ids"][ok])
        assert np.allclose(got["nuc_probs"][ok][m], tr["nuc_probs"][ok][m], rtol=1e-5)
    return got, fx, tr


# ---------------------------------------------------------------- building blocks

def test_expneg_bit_exact(oracle, rocm):
    from born_amd import _capi
    d = np.concatenate([np.linspace(0, 90, 20001), np.random.default_rng(0).uniform(0, 40, 50000),
                        [0.0, 80.0, 80.00001, np.inf]]).astype(np.float32)
    buf_in = rocm.DeviceBuffer.from_numpy(d)
    buf_out = rocm.DeviceBuffer(d.nbytes)
    _capi.check(_capi.lib().born_rocm_expneg(buf_in.ptr, buf_out.ptr, d.size, None))
    got = buf_out.to_numpy(np.float32, d.shape)
    want = oracle.expneg(d)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


def test_uniform_stream_bit_exact(oracle, rocm):
    from born_amd import _capi
    n = 1000
    out = rocm.DeviceBuffer(4 * n)
    for seed, step in [(0, 0), (1234, 7), (-5, 3)]:
        _capi.check(_capi.lib().born_rocm_uniforms(seed, step, out.ptr, n, None))
        got = out.to_numpy(np.float32, (n,))
        want = np.array([oracle.uniform(seed, step, r) for r in range(n)], dtype=np.float32)
        assert np.array_equal(got, want)
        assert got.min() >= 0.0 and got.max() < 1.0


# ---------------------------------------------------------------- reference-pinned operators

def _argmax(rocm, x, stride=None):
    B, V = x.shape
    s = rocm.NewSampler(max_batch=B, max_vocab=V)
    if stride:
        xp = np.zeros((B, stride), np.float32)
        xp[:, :V] = x
        xp[:, V:] = 1e30              # padding must never be read as data
        d = rocm.DeviceBuffer.from_numpy(xp)
    else:
        d = rocm.DeviceBuffer.from_numpy(x)
    t = rocm.DeviceBuffer(4 * B)
    s.Argmax(d, B, V, t, row_stride=stride)
    s.Argmax(d, B, V, t, row_stride=stride)       # second launch: the workspace of the first is reused
    return t.to_numpy(np.int32, (B,))


def test_argmax_reference_kats_and_tie_rule(oracle, rocm):
    x = np.array([[1, 2, 3], [3, 1, 2], [2, 3, 1], [1, 1, 3]], dtype=np.float32)        # TestAccuracy vectors
    assert _argmax(rocm, x).tolist() == [2, 0, 1, 2]
    x = np.array([[5, 5, 5], [1, 7, 7], [np.nan, 9, 1], [1, np.nan, 0], [-np.inf, -np.inf, -np.inf]], dtype=np.float32)
    assert _argmax(rocm, x).tolist() == oracle.argmax_ref(x).tolist() == [0, 1, 0, 0, 0]
    assert _argmax(rocm, np.tile(x, (16, 1))).tolist() == [0, 1, 0, 0, 0] * 16         # 80 rows: the row-per-workgroup kernel
    wide = np.full((64, 9000), -np.inf, np.float32)
    wide[1, 8999] = 3.0; wide[2, 0] = np.nan; wide[2, 5] = 9.0; wide[3, 4096:4100] = 7.0; wide[4, :] = np.nan
    assert _argmax(rocm, wide).tolist() == oracle.argmax_ref(wide).tolist()


@pytest.mark.parametrize("B,V,stride", [(64, 32000, None), (7, 8193, None), (5, 1001, 1003), (3, 128256, None), (2, 5, 8),
                                        (63, 32000, None), (64, 8193, None), (70, 1001, 1003), (65, 5, 8), (64, 16384, 16388),
                                        (96, 128256, None), (64, 1, None), (64, 20001, 20004),
                                        (67, 4096, None), (66, 4097, None), (301, 1024, None), (130, 16384, None), (65, 16385, 16388),
                                        (1000, 63, 64), (70, 4095, 4095), (4000, 10, None), (300, 16, 19), (77, 17, None), (129, 64, None),
                                        (64, 65, None)])
def test_argmax_random_and_ties(oracle, rocm, B, V, stride):
    rng = np.random.default_rng(V)
    x = rng.standard_normal((B, V), dtype=np.float32)
    assert np.array_equal(_argmax(rocm, x, stride), oracle.argmax_ref(x))
    xi = rng.integers(-2, 3, size=(B, V)).astype(np.float32)                              # thousands of ties
    assert np.array_equal(_argmax(rocm, xi, stride), oracle.argmax_ref(xi))


def test_softmax_operators(oracle, rocm):
    import json, os
    with open(os.path.join(os.path.dirname(__file__), "golden", "reference_kats.json")) as f:
        kats = json.load(f)
    s = rocm.NewSampler(max_batch=64, max_vocab=32000)

    def soft(x, log=False):
        B, V = x.shape
        d, o = rocm.DeviceBuffer.from_numpy(x), rocm.DeviceBuffer(x.nbytes)
        s.Softmax(d, B, V, o, log=log)
        return o.to_numpy(np.float32, x.shape)

    for case in kats["softmax"]:
        x = np.array(case["input"], dtype=np.float32)
        got = soft(x).astype(np.float64)
        want = oracle.softmax_ref(x).astype(np.float64)          # the reference's arithmetic
        assert np.max(np.abs(got - want)) <= 1e-6, case["source"]
        assert abs(got.sum() - 1.0) <= 1e-6 and np.all(np.isfinite(got))
    for case in kats["log_softmax"]:
        x = np.array(case["input"], dtype=np.float32)
        got = soft(x, log=True).astype(np.float64)
        assert np.all(np.isfinite(got))
        assert np.max(np.abs(got - oracle.log_softmax_ref(x))) <= 1e-4 * max(1.0, np.abs(x).max() * 1e-2)
    rng = np.random.default_rng(1)
    x = (rng.standard_normal((64, 32000), dtype=np.float32) * 2).astype(np.float32)
    got = soft(x)
    want = oracle.softmax_f64(x)
    assert np.allclose(got, want, rtol=1e-5, atol=1e-30)
    assert np.max(np.abs(got - oracle.softmax_ref(x))) <= 1e-6
    lg = soft(x, log=True).astype(np.float64)
    assert np.max(np.abs(lg - np.log(want))) < 1e-5


@pytest.mark.parametrize("B,V,pad", [(5, 1, 0), (7, 3, 0), (33, 64, 0), (1000, 10, 0), (300, 16, 1), (77, 17, 0), (129, 63, 2), (64, 65, 0), (6, 256, 0), (600, 257, 0), (9, 512, 4), (9, 513, 1), (300, 1000, 0),
                                     (17, 1024, 0), (17, 1025, 0), (9, 2048, 0), (9, 2049, 3), (260, 4096, 8), (7, 4097, 0), (5, 8192, 4),
                                     (5, 8193, 0), (3, 16384, 0), (3, 16385, 2), (3, 32768, 0), (3, 32769, 1), (4, 70001, 0), (2, 128256, 0)])
def test_softmax_every_row_length_and_layout(oracle, rocm, B, V, pad):
    # One wave, 256 or 1024 lanes per row with the row held in registers, or three sweeps, by the row's length; rows that
    # start unaligned (a pitch that is no multiple of four) and ragged ends take the element-wise loads and stores.
    # Held to 1e-5 of the fp64 softmax; and equal, bit for bit, to the kernel's own definition put together from the
    # oracle's pieces: fl32(fl64(e) / Z) with e the oracle's expneg of (max - z) and Z the sum of trunc(e * 2^S) * 2^-S.
    rng = np.random.default_rng(B * 7919 + V)
    x = (rng.standard_normal((B, V + pad)) * 3.0).astype(np.float32)
    if V > 8:
        x[0, rng.integers(0, V, size=3)] = -np.inf
        x[B - 1, rng.integers(0, V, size=2)] = np.float32(-3e38)
        x[B // 2, :V] = np.round(x[B // 2, :V])                             # ties at the maximum
    s = rocm.NewSampler(max_batch=B, max_vocab=V)
    d, o = rocm.DeviceBuffer.from_numpy(x), rocm.DeviceBuffer(4 * B * V)
    rows = x[:, :V]
    for log in (False, True):
        s.Softmax(d, B, V, o, row_stride=V + pad, log=log)
        got = o.to_numpy(np.float32, (B, V))
        want = oracle.softmax_f64(np.ascontiguousarray(rows))
        if log:
            fin = want > 0
            assert np.max(np.abs(got[fin].astype(np.float64) - np.log(want[fin]))) < 2e-5 and np.all(got[~fin] < -80.0)
            continue
        assert np.allclose(got, want, rtol=1e-5, atol=1e-30)
        assert np.all(np.abs(got.sum(axis=1, dtype=np.float64) - 1.0) < 1e-5)
        m, Zi = oracle.row_stats(np.ascontiguousarray(rows))                # the oracle's maximum and integer normaliser
        assert np.array_equal(m, rows.max(axis=1))
        with np.errstate(invalid="ignore"):
            dist = (m[:, None] - rows).astype(np.float32)
        dist[rows == m[:, None]] = 0.0
        e = oracle.expneg(dist)
        Z = Zi.astype(np.float64) * 2.0 ** -(62 - int(V).bit_length())       # (2^S with S = 62 - bits(V): a row sums below 2^62)
        assert np.array_equal(got.view(np.uint32), (e.astype(np.float64) / Z[:, None]).astype(np.float32).view(np.uint32))
    s.Close()


# ---------------------------------------------------------------- sampling: single-pass top-k kernel
# path 0 = the default kernel selection (1 <= top_k <= 512: one workgroup per row, one launch); path 2 = the same with
# the 512-thread instance (top_k <= 128) whatever the batch, which by default only batches of more rows than CUs get

TOPK_PATHS = [0, 2]


@pytest.mark.parametrize("path", TOPK_PATHS)
@pytest.mark.parametrize("B,V,T,k,p,rep,H", [
    (1, 32000, 0.8, 40, 0.95, 1.1, 64),          # C1 shape
    (32, 128256, 0.7, 50, 0.9, 1.15, 512),       # C3 shape, 32 rows
    (16, 32000, 1.0, 1, 1.0, 1.3, 16),           # greedy with penalty
    (16, 8192, 1.3, 64, 0.5, 1.0, 0),
    (16, 8193, 0.5, 7, 1.0, 0.8, 8),             # tail segment of one element; penalty < 1 boosts
    (9, 1000, 1.0, 50, 0.9, 1.2, 300),           # fewer lanes than logits per wave
    (9, 777, 0.9, 64, 0.99, 1.5, 2000),          # history longer than the vocabulary
    (4, 100, 1.0, 64, 0.9, 1.1, 10),
    (4, 3, 1.0, 2, 0.9, 1.0, 0),
    (32, 128256, 0.7, 128, 0.9, 1.15, 512),      # two survivors per lane of the last wave
    (16, 32000, 1.0, 65, 1.0, 1.0, 0),           # 65: one lane holds a second survivor
    (16, 50257, 1.1, 100, 0.95, 1.2, 1500),      # history longer than the workgroup
    (9, 777, 0.9, 127, 0.99, 1.5, 2000),
    (4, 200, 1.0, 128, 0.9, 1.1, 10),            # a row of one wave: no first-stage threshold for top_k > 64
    (4, 129, 0.8, 128, 0.7, 1.0, 0),
    (32, 128256, 0.7, 129, 0.9, 1.15, 512),      # beyond 128: ranked through buckets, four survivors per lane
    (32, 128256, 0.7, 256, 0.9, 1.15, 512),
    (32, 128256, 0.7, 512, 0.9, 1.15, 512),      # eight survivors per lane
    (16, 32000, 1.0, 257, 1.0, 1.0, 0),
    (16, 50257, 1.1, 400, 0.95, 1.2, 1500),      # history longer than the workgroup
    (9, 2000, 0.9, 512, 0.99, 1.5, 3000),        # a quarter of the vocabulary survives the cut
    (9, 777, 0.9, 300, 0.99, 1.5, 2000),
    (4, 600, 0.8, 512, 0.7, 1.0, 0),             # a row of three waves: no first-stage threshold
    (6, 16385, 0.7, 333, 0.9, 1.3, 64),          # one element in the second stage
    (32, 128256, 0.7, 50, 0.9, 0.8, 512),        # a penalty < 1 raises logits: seen ids join the candidates from the history's hash
    (16, 32000, 1.0, 100, 0.95, 0.5, 1000),
    (16, 32000, 1.3, 300, 0.9, 0.25, 1024),      # the longest history the hash takes
    (16, 50257, 1.1, 256, 0.95, 0.7, 1500),      # beyond it: the general kernel
])
def test_topk_kernel_against_oracle(oracle, rocm, B, V, T, k, p, rep, H, path):
    rng = np.random.default_rng(B * 1000003 + V)
    x = (rng.standard_normal((B, V), dtype=np.float32) * np.float32(1.5)).astype(np.float32)
    u = rng.random(B, dtype=np.float32)
    hist = ((rng.zipf(1.1, size=(B, H)) - 1) % V).astype(np.int32) if H else None
    got, _, _ = _check_against_oracle(oracle, rocm, x, u, T, k, p, rep, hist, nuc=min(512, max(k, 1)), path=path)
    c = got["counters"]
    if rep < 1.0 and H > 1024:   # a boosting penalty over a history longer than the workgroup's hash is served by the general kernel
        assert c["general_rows"] == B
    else:
        assert c["topk_rows"] + c["fallback_rows"] == B and c["general_rows"] == 0


@pytest.mark.parametrize("B,V,k,H", [(300, 20000, 50, 64), (257, 8193, 128, 700), (600, 3001, 7, 0), (520, 16384, 100, 512)])
def test_topk_kernel_more_rows_than_compute_units(oracle, rocm, B, V, k, H):
    # Batches of more rows than the device has CUs run the 512-thread instance of the kernel (two rows to a CU at a
    # time) by the default selection; same tokens, same probabilities, every row settled by the single-pass kernel.
    rng = np.random.default_rng(B + V)
    x = (rng.standard_normal((B, V), dtype=np.float32) * np.float32(1.5)).astype(np.float32)
    x[::7] = np.sort(x[::7], axis=1)                                     # some rows ascending: thresholds raised by the waves
    u = rng.random(B, dtype=np.float32)
    hist = ((rng.zipf(1.1, size=(B, H)) - 1) % V).astype(np.int32) if H else None
    got, _, _ = _check_against_oracle(oracle, rocm, x, u, 0.7, k, 0.9, 1.15, hist, nuc=k)
    c = got["counters"]
    assert c["topk_rows"] + c["fallback_rows"] == B and c["general_rows"] == 0


@pytest.mark.parametrize("V,H", [(128256, 512), (32000, 1000), (5003, 64), (777, 1024)])
def test_topk_kernel_penalties_that_raise_logits(oracle, rocm, V, H):
    # A repetition penalty below 1 and negative frequency / presence penalties lift seen ids from far below the
    # streamed threshold into the top_k (and past the maximum); each seen id must be ranked by its penalised logit
    # exactly once, whether its stored logit was listed or not.
    rng = np.random.default_rng(V + H)
    B = 24
    x = (rng.standard_normal((B, V), dtype=np.float32) * np.float32(2.0)).astype(np.float32)
    u = rng.random(B, dtype=np.float32)
    hist = ((rng.zipf(1.2, size=(B, H)) - 1) % V).astype(np.int32)
    hist[:, : H // 4] = rng.integers(0, V, size=(B, H // 4))            # a quarter spread over the vocabulary
    for r in range(B):                                                   # some rows: the history holds the row's largest logits too
        if r % 3 == 0:
            hist[r, :8] = np.argsort(-x[r])[:8]
    x[1, hist[1, :50]] = -np.inf                                         # seen ids that stay impossible
    x[2, hist[2, :50]] = np.nan
    hl = rng.integers(0, H + 1, size=B).astype(np.int32)
    hl[:4] = H
    for (T, k, p, rep, freq, pres) in [(0.8, 50, 0.9, 0.5, 0.0, 0.0), (1.0, 128, 1.0, 0.1, 0.0, 0.0), (1.2, 300, 0.95, 1.0, -0.5, -1.0),
                                       (0.7, 40, 0.9, 1.3, -3.0, 0.0), (1.0, 1, 1.0, 0.7, 0.0, -2.0), (1.0, 64, 0.99, 0.9, -0.1, 0.3)]:
        if k >= V:
            continue
        got, _, _ = _check_against_oracle(oracle, rocm, x, u, T, k, p, rep, hist, hl, nuc=min(512, k), freq=freq, pres=pres)
        c = got["counters"]
        assert c["general_rows"] == 0 and c["topk_rows"] + c["fallback_rows"] == B
        if V > 20000:
            assert c["fallback_rows"] <= 2, (T, k, p, rep, freq, pres, c)   # (the NaN / -inf rows may need the exact selection)


@pytest.mark.parametrize("path", TOPK_PATHS)
def test_topk_kernel_hist_len_and_strided_rows(oracle, rocm, path):
    rng = np.random.default_rng(5)
    B, V, H = 12, 5000, 40
    x = rng.standard_normal((B, V), dtype=np.float32)
    u = rng.random(B, dtype=np.float32)
    hist = rng.integers(0, V, size=(B, H)).astype(np.int32)
    hl = rng.integers(0, H + 1, size=B).astype(np.int32)
    _check_against_oracle(oracle, rocm, x, u, 0.9, 20, 0.9, 1.4, hist, hl, path=path)
    # unaligned row stride (scalar load path): rows placed in a wider buffer
    s = rocm.NewSampler(rocm.SamplerConfig(Temperature=0.9, TopK=20, TopP=0.9), max_batch=B, max_vocab=V)
    s.SetPath(path)
    xp = np.full((B, V + 3), 99.0, np.float32)
    xp[:, :V] = x
    d_x, d_u, d_t = rocm.DeviceBuffer.from_numpy(xp), rocm.DeviceBuffer.from_numpy(u), rocm.DeviceBuffer(4 * B)
    s.Sample(d_x, B, V, None, None, d_u, d_t, row_stride=V + 3)
    want = oracle.sample(x, u, 0.9, 20, 0.9, mode=oracle.MODE_FIXED)["tokens"]
    assert np.array_equal(d_t.to_numpy(np.int32, (B,)), want)


@pytest.mark.parametrize("path", TOPK_PATHS)
def test_topk_kernel_ties_and_special_values(oracle, rocm, path):
    rng = np.random.default_rng(6)
    B, V = 24, 20000
    xi = rng.integers(-3, 4, size=(B, V)).astype(np.float32)           # thousands of exact ties at the cut
    u = rng.random(B, dtype=np.float32)
    got, _, _ = _check_against_oracle(oracle, rocm, xi, u, 0.7, 50, 0.9, nuc=64, path=path)
    assert got["counters"]["fallback_rows"] > 0                         # ties overflow the single-pass path
    x = rng.standard_normal((B, V), dtype=np.float32)
    x[:, ::7] = -np.inf
    x[:, 5::11] = np.nan
    x[0, 100] = np.inf
    x[1, :] = -np.inf                                                   # nothing finite: uniform over ids
    x[2, 17:] = -np.inf                                                 # fewer finite logits than top_k
    x[3, :] = 0.0
    x[3, 1::2] = -0.0                                                   # -0 ties with +0
    _check_against_oracle(oracle, rocm, x, u, 1.0, 40, 0.95, nuc=64, path=path)


def _shaped_rows(kind, B, V, rng):
    """Rows whose large values sit where a threshold that tightens while the row streams is most easily
    wrong: late in the row, in a narrow band, in huge ranges, or tied across the cut."""
    i = np.arange(V, dtype=np.float64)
    if kind == "ascending":                 # every later stage beats everything before it
        x = np.tile(i / V * 20 - 10, (B, 1)) + rng.standard_normal((B, V)) * 1e-3
    elif kind == "descending":              # the first stage already holds the whole answer
        x = np.tile(10 - i / V * 20, (B, 1)) + rng.standard_normal((B, V)) * 1e-3
    elif kind == "late_step":               # the answer lies wholly in the last tenth of the row
        x = rng.standard_normal((B, V))
        x[:, V - V // 10:] += 30
    elif kind == "late_few":                # a handful of winners at the very end, nothing close to them
        x = rng.standard_normal((B, V))
        x[:, -37:] += 12
    elif kind == "cauchy":                  # a range of 1e6 and more between neighbours in order
        x = rng.standard_cauchy((B, V)) * 3
    elif kind == "narrow":                  # the whole row within a few hundred ulps
        x = 5.0 + rng.integers(0, 300, size=(B, V)) * 2.0 ** -21
    elif kind == "few_values":              # a dozen distinct values: ties across every cut
        x = rng.integers(0, 12, size=(B, V)) * 0.37 - 2
    elif kind == "negative_huge":           # large negative magnitudes: order keys far from the float's own order
        x = -np.abs(rng.standard_normal((B, V))) * 1e30
    elif kind == "rising_blocks":           # each block of 4096 a little higher than the last one
        x = rng.standard_normal((B, V)) + (np.arange(V) // 4096) * 0.5
    elif kind == "mid_bump":                # the answer lies wholly in a tenth of the row around its middle
        x = rng.standard_normal((B, V))
        x[:, V // 2:V // 2 + V // 10] += 30
    elif kind == "log_probs":               # all negative, one token close to certain: keys crowd around zero
        x = -np.abs(rng.standard_normal((B, V))) * 4 - 3
        x[np.arange(B), rng.integers(0, V, B)] = -1e-6
        x = np.sort(x, axis=1)                  # ... and sorted ascending
    else:
        raise ValueError(kind)
    return x.astype(np.float32)


@pytest.mark.parametrize("kind", ["ascending", "descending", "late_step", "late_few", "cauchy", "narrow", "few_values",
                                  "negative_huge", "rising_blocks", "mid_bump", "log_probs"])
@pytest.mark.parametrize("V,pad", [(49152, 0), (49153, 3), (65537, 0), (128256, 0), (151937, 7), (393216, 0)])
def test_topk_kernel_rows_that_stress_the_streamed_threshold(oracle, rocm, kind, V, pad):
    """The single-pass kernel raises its threshold while the row streams. Whatever the shape of the row, the
    result is the oracle's, bit for bit: either the single pass proves its candidate set or the row falls back;
    without ties and without a penalty that moves the winners it must not fall back."""
    rng = np.random.default_rng([len(kind), ord(kind[0]), ord(kind[-1]), V])
    B, H = 6, 96
    x = _shaped_rows(kind, B, V, rng)
    u = rng.random(B, dtype=np.float32)
    top = np.argsort(-x, axis=1, kind="stable")[:, :H // 2].astype(np.int32)      # half the history penalises the winners
    hist = np.concatenate([top, rng.integers(0, V, size=(B, H - H // 2)).astype(np.int32)], axis=1)
    for k, p, rep in [(50, 0.9, 1.3), (128, 1.0, 1.0), (1, 1.0, 2.0), (300, 0.95, 1.2)]:
        want = oracle.sample(x, u, 0.7, k, p, rep, hist if rep != 1.0 else None, mode=oracle.MODE_FIXED, nuc_cap=min(k, 64))
        s = rocm.NewSampler(rocm.SamplerConfig(Temperature=0.7, TopK=k, TopP=p, RepetitionPenalty=rep), max_batch=B, max_vocab=V)
        xp = np.full((B, V + pad), 1e38, np.float32)                                  # padding must never be read as data
        xp[:, :V] = x
        d_x, d_u, d_t, d_p = rocm.DeviceBuffer.from_numpy(xp), rocm.DeviceBuffer.from_numpy(u), rocm.DeviceBuffer(4 * B), rocm.DeviceBuffer(4 * B)
        d_h = rocm.DeviceBuffer.from_numpy(hist) if rep != 1.0 else None
        s.Sample(d_x, B, V, d_h, None, d_u, d_t, probs_out=d_p, row_stride=V + pad, hist_stride=H if rep != 1.0 else 0)
        s.Status()
        c = s.Counters()
        s.Close()
        assert c["topk_rows"] + c["fallback_rows"] == B and c["general_rows"] == 0
        # Wherever the large logits sit, the single pass settles the row itself: the last stage is examined second and a
        # wave whose list overflows raises its own threshold.  (Not asserted: rows of equal logits by the thousand, and
        # the configurations whose history penalises the row's winners, which the proof hands to the exact selection.)
        if rep == 1.0 and kind not in ("narrow", "few_values", "log_probs"):     # (log_probs: still falls back at some sizes)
            assert c["fallback_rows"] == 0, (kind, V, k, c)
        assert np.array_equal(d_t.to_numpy(np.int32, (B,)), want["tokens"]), (kind, V, k)
        assert np.array_equal(d_p.to_numpy(np.float32, (B,)).view(np.uint32), want["probs"].view(np.uint32)), (kind, V, k)


@pytest.mark.parametrize("path", TOPK_PATHS)
def test_topk_and_general_kernels_agree(oracle, rocm, path):
    rng = np.random.default_rng(7)
    B, V, H = 24, 40000, 128
    x = (rng.standard_normal((B, V), dtype=np.float32) * 2).astype(np.float32)
    u = rng.random(B, dtype=np.float32)
    hist = rng.integers(0, V, size=(B, H)).astype(np.int32)
    a = _run(rocm, x, u, 0.7, 50, 0.9, 1.15, hist, nuc=64, path=path)
    b = _run(rocm, x, u, 0.7, 50, 0.9, 1.15, hist, nuc=64, path=1)
    assert a["counters"]["topk_rows"] == B and b["counters"]["general_rows"] == B
    for key in ("tokens", "n_nucleus", "nuc_ids"):
        assert np.array_equal(a[key], b[key]), key
    assert np.array_equal(a["probs"].view(np.uint32), b["probs"].view(np.uint32))


def test_kernel_selection_by_shape(oracle, rocm):
    """A vocabulary beyond the single-pass kernel's limit takes the general kernel; no top-k cut takes the
    three-sweep kernel; a general-kernel run of the same input agrees bit for bit."""
    rng = np.random.default_rng(17)
    B, V = 2, 400000
    x = (rng.standard_normal((B, V), dtype=np.float32) * 2).astype(np.float32)
    u = rng.random(B, dtype=np.float32)
    hist = rng.integers(0, V, size=(B, 64)).astype(np.int32)
    got, _, _ = _check_against_oracle(oracle, rocm, x, u, 0.9, 50, 0.9, 1.2, hist, nuc=64)
    assert got["counters"]["general_rows"] == B and got["counters"]["topk_rows"] == 0
    a = _run(rocm, x, u, 0.9, 0, 0.9, 1.2, hist, path=0)
    b = _run(rocm, x, u, 0.9, 0, 0.9, 1.2, hist, path=1)
    assert np.array_equal(a["tokens"], b["tokens"]) and np.array_equal(a["probs"].view(np.uint32), b["probs"].view(np.uint32))


# ---------------------------------------------------------------- sampling: kernel without a top-k cut (path 0, top_k 0)
# and the general kernel (path 0 for top_k > 512, path 1 for everything)

@pytest.mark.parametrize("path", [0, 1, 2])
@pytest.mark.parametrize("B,V,T,k,p,rep,H", [
    (64, 32000, 1.0, 0, 1.0, 1.0, 0),            # C2 multinomial shape
    (16, 152064, 1.2, 0, 0.99, 1.05, 2048),      # C5 shape, 16 rows
    (16, 32000, 0.9, 700, 0.9, 1.1, 64),         # top_k above the single-pass limit
    (8, 50000, 1.0, 20000, 0.8, 1.0, 0),         # top_k too large to list: count descent
    (8, 50000, 1.0, 20000, 1.0, 1.0, 0),
    (16, 4097, 0.6, 0, 0.3, 1.0, 0),
    (16, 1000, 2.0, 600, 1.0, 1.2, 50),
    (5, 2, 1.0, 0, 0.9, 1.0, 0),
    (5, 1, 1.0, 0, 0.9, 1.0, 0),
])
def test_general_kernel_against_oracle(oracle, rocm, B, V, T, k, p, rep, H, path):
    rng = np.random.default_rng(B * 7919 + V + k)
    x = rng.standard_normal((B, V), dtype=np.float32)
    u = rng.random(B, dtype=np.float32)
    hist = rng.integers(0, V, size=(B, H)).astype(np.int32) if H else None
    got, _, _ = _check_against_oracle(oracle, rocm, x, u, T, k, p, rep, hist, path=path)
    assert got["counters"]["general_rows"] == B


@pytest.mark.parametrize("path", [0, 1, 2])
def test_general_kernel_degenerate_rows(oracle, rocm, path):
    rng = np.random.default_rng(8)
    B, V = 12, 30000
    u = rng.random(B, dtype=np.float32)
    x = np.zeros((B, V), np.float32)                                    # every logit equal: radix descent on ids
    got, _, _ = _check_against_oracle(oracle, rocm, x, u, 1.0, 0, 1.0, path=path)
    if path != 1:
        assert got["counters"]["fallback_rows"] == B                    # ... taken by the kernel without a top-k cut
    _check_against_oracle(oracle, rocm, x, u, 1.0, 0, 0.5, path=path)
    _check_against_oracle(oracle, rocm, x, u, 1.0, 9000, 0.9, path=path)
    xi = rng.integers(-1, 2, size=(B, V)).astype(np.float32)            # three values
    _check_against_oracle(oracle, rocm, xi, u, 0.8, 0, 0.9, path=path)
    _check_against_oracle(oracle, rocm, xi, u, 0.8, 12345, 0.9, path=path)
    x = rng.standard_normal((B, V), dtype=np.float32)
    x[:, ::3] = -np.inf
    x[:, 1::5] = np.nan
    x[0, :] = -np.inf
    x[1, 7] = np.inf
    _check_against_oracle(oracle, rocm, x, u, 1.0, 0, 0.95, path=path)
    far = rng.standard_normal((B, V), dtype=np.float32) - 200.0         # everything but one far below the maximum
    far[:, 11] = 0.0
    _check_against_oracle(oracle, rocm, far, u, 1.0, 0, 1.0, path=path)


# ---------------------------------------------------------------- min-p

@pytest.mark.parametrize("path", [0, 1, 2])
@pytest.mark.parametrize("B,V,T,k,p,rep,H,min_p", [
    (32, 128256, 0.7, 50, 0.9, 1.15, 512, 0.05),    # C3 shape with min-p: single-pass top-k kernel
    (16, 32000, 1.0, 40, 1.0, 1.0, 0, 0.1),         # min-p is the only cut inside the top-k
    (16, 32000, 1.0, 64, 1.0, 1.1, 32, 0.5),        # few survivors
    (16, 32000, 1.0, 0, 1.0, 1.0, 0, 0.02),         # no top-k: nucleus kernel, min-p alone
    (16, 152064, 1.2, 0, 0.95, 1.05, 2048, 0.01),   # C5 shape with min-p
    (16, 32000, 0.9, 500, 0.9, 1.1, 64, 0.05),      # general kernel, top-k counted
    (8, 50000, 1.0, 20000, 1.0, 1.0, 0, 0.001),     # general kernel, top-k by count descent
    (8, 4097, 2.0, 0, 0.5, 1.0, 0, 0.2),
    (5, 2, 1.0, 0, 1.0, 1.0, 0, 0.3),
    (5, 1, 1.0, 0, 1.0, 1.0, 0, 0.9),
    (8, 1000, 1.0, 10, 0.9, 1.0, 0, 1e-30),         # a bound beyond every mass: as if off
])
def test_min_p_against_oracle(oracle, rocm, B, V, T, k, p, rep, H, min_p, path):
    rng = np.random.default_rng(B * 7919 + V + int(min_p * 1000))
    x = (rng.standard_normal((B, V), dtype=np.float32) * np.float32(2.0)).astype(np.float32)
    u = rng.random(B, dtype=np.float32)
    hist = ((rng.zipf(1.1, size=(B, H)) - 1) % V).astype(np.int32) if H else None
    nuc = k if 1 <= k <= 512 else 0
    _, fx, _ = _check_against_oracle(oracle, rocm, x, u, T, k, p, rep, hist, nuc=nuc, path=path, min_p=min_p)
    if nuc and min_p >= 0.05:
        assert (fx["n_nucleus"] < k).any(), "the case is meant to have min-p bind"


def test_min_p_survivor_set_and_special_rows(oracle, rocm):
    # probabilities 1/2, 1/4, 1/8, 1/16, 1/16: the ratio to the top is 1, 1/2, 1/4, 1/8, 1/8
    # (and a sixth entry far below, so that top_k = 5 is a real cut and the nucleus gets listed)
    x = np.log(np.array([[0.5, 0.25, 0.125, 0.0625, 0.0625, 1e-12]] * 4, dtype=np.float64)).astype(np.float32)
    u = np.array([0.0, 0.4, 0.8, 0.999], dtype=np.float32)
    for min_p, n in [(0.1, 5), (0.2, 3), (0.3, 2), (0.6, 1)]:
        got = _run(rocm, x, u, k=5, nuc=5, min_p=min_p)
        assert (got["n_nucleus"] == n).all(), (min_p, got["n_nucleus"])
        assert (got["tokens"] < n).all()
        want = np.array([0.5, 0.25, 0.125, 0.0625, 0.0625][:n]) / sum([0.5, 0.25, 0.125, 0.0625, 0.0625][:n])
        assert np.allclose(got["nuc_probs"][:, :n], want, rtol=1e-6)
        assert (got["nuc_ids"][:, n:] == -1).all()
    # masked rows: -inf everywhere but two entries; all -inf (every entry ties at the maximum and stays)
    y = np.full((2, 1000), -np.inf, dtype=np.float32)
    y[0, 17] = 1.0
    y[0, 900] = 0.0
    for path in (0, 1):
        for k in (0, 8):
            _check_against_oracle(oracle, rocm, y, np.array([0.9, 0.5], dtype=np.float32), k=k, path=path, min_p=0.5)


def test_min_p_is_validated(rocm):
    for bad in (-0.1, 1.0, 1.5, float("nan")):
        with pytest.raises(rocm.SamplerPanic, match="min_p"):
            rocm.NewSampler(rocm.SamplerConfig(MinP=bad), max_batch=1, max_vocab=16)
    s = rocm.NewSampler(rocm.SamplerConfig(MinP=0.25), max_batch=1, max_vocab=16)
    assert s.Config().MinP == 0.25
    s.Close()


# ---------------------------------------------------------------- frequency and presence penalties

@pytest.mark.parametrize("path", [0, 1, 2])
@pytest.mark.parametrize("B,V,T,k,p,rep,H,freq,pres,route", [
    (32, 128256, 0.7, 50, 0.9, 1.15, 512, 0.3, 0.5, "topk"),     # C3 shape: single-pass kernel, history hashed
    (16, 32000, 1.0, 40, 0.95, 1.0, 64, 0.5, 0.0, "topk"),       # frequency alone, no repetition penalty
    (16, 32000, 1.0, 40, 0.95, 1.0, 64, 0.0, 1.5, "topk"),       # presence alone
    (9, 8000, 0.9, 64, 0.99, 1.2, 3000, 0.2, 0.3, "topk"),       # history longer than 1024: candidates are hashed instead
    (16, 32000, 1.0, 20, 0.9, 1.1, 128, -0.4, 0.2, "topk"),      # a negative penalty raises logits: seen ids join the candidates
    (16, 32000, 1.0, 20, 0.9, 1.1, 1024, -0.4, -0.2, "topk"),
    (16, 32000, 1.0, 20, 0.9, 1.1, 1025, -0.4, 0.2, "general"),  # ... a history beyond the hash: the general kernel
    (16, 32000, 1.0, 0, 1.0, 1.0, 256, 0.4, 0.4, "nucleus"),     # no top-k: three-sweep kernel
    (16, 152064, 1.2, 0, 0.99, 1.05, 2048, 0.1, 0.6, "nucleus"), # C5 shape
    (16, 32000, 0.9, 500, 0.9, 1.1, 64, 0.25, 0.25, "topk"),       # beyond 128: the single-pass kernel's larger sizes
    (16, 32000, 0.9, 700, 0.9, 1.1, 64, 0.25, 0.25, "general"),
    (8, 50000, 1.0, 20000, 0.8, 1.0, 300, 0.5, 0.5, "general"),
    (8, 1001, 1.0, 0, 0.9, 1.0, 5000, 0.05, 1.0, "nucleus"),     # unaligned rows, history much longer than the vocabulary
    (8, 1001, 1.0, 10, 0.9, 1.0, 5000, 0.05, 1.0, "topk"),
    (12, 50257, 0.8, 100, 0.95, 1.1, 4096, 0.02, 0.4, "topk"),    # the longest history counted inside the kernel
    (12, 50257, 0.8, 100, 0.95, 1.1, 4097, 0.02, 0.4, "topk"),    # one more: the table of counts
    (16, 32000, 1.0, 40, 0.95, 1.0, 1024, 0.5, 0.1, "topk"),      # the longest history hashed whole
    (16, 32000, 1.0, 40, 0.95, 1.0, 1025, 0.5, 0.1, "topk"),
])
def test_frequency_and_presence_penalties_against_oracle(oracle, rocm, B, V, T, k, p, rep, H, freq, pres, route, path):
    rng = np.random.default_rng(B * 104729 + V + H)
    x = (rng.standard_normal((B, V), dtype=np.float32) * np.float32(1.5)).astype(np.float32)
    u = rng.random(B, dtype=np.float32)
    hist = ((rng.zipf(1.2, size=(B, H)) - 1) % V).astype(np.int32)        # heavy repeats of the small ids
    x[:, :8] += np.float32(4.0)                                             # ... which are also the likely tokens
    hist_len = rng.integers(H // 2, H + 1, size=B).astype(np.int32)
    nuc = k if 1 <= k <= 512 else 0
    got, fx, _ = _check_against_oracle(oracle, rocm, x, u, T, k, p, rep, hist, hist_len, nuc=nuc, path=path, freq=freq, pres=pres)
    plain = oracle.sample(x, u, T, k, p, rep, hist, hist_len, mode=oracle.MODE_FIXED)
    assert (plain["tokens"] != fx["tokens"]).any() or not np.array_equal(plain["probs"], fx["probs"]), "the penalties are meant to matter"
    c = got["counters"]
    if path != 1 and route == "topk":
        assert c["topk_rows"] + c["fallback_rows"] == B and c["general_rows"] == 0
    if path != 1 and route == "general":
        assert c["general_rows"] == B


def test_frequency_penalty_table_is_clean_between_calls(oracle, rocm):
    # one handle, three calls with different histories and shapes: each equals a fresh evaluation by the oracle
    rng = np.random.default_rng(77)
    Bm, Vm = 24, 40000
    s = rocm.NewSampler(rocm.SamplerConfig(TopK=30, TopP=0.9, RepetitionPenalty=1.1, FrequencyPenalty=0.4, PresencePenalty=0.3),
                        max_batch=Bm, max_vocab=Vm)
    for (B, V, H) in [(24, 40000, 700), (10, 32000, 100), (24, 40000, 1500), (5, 999, 50)]:
        x = (rng.standard_normal((B, V), dtype=np.float32) * np.float32(1.5)).astype(np.float32)
        x[:, :8] += np.float32(4.0)
        u = rng.random(B, dtype=np.float32)
        hist = ((rng.zipf(1.2, size=(B, H)) - 1) % V).astype(np.int32)
        got = rocm.sample_host(s, x, u, hist)
        fx = oracle.sample(x, u, 1.0, 30, 0.9, 1.1, hist, mode=oracle.MODE_FIXED, freq=0.4, pres=0.3)
        assert np.array_equal(got["tokens"], fx["tokens"]), (B, V, H)
        assert np.array_equal(got["probs"].view(np.uint32), fx["probs"].view(np.uint32))
    # switching the penalties on later allocates the table then; switching them off stops using it
    t = rocm.NewSampler(rocm.SamplerConfig(TopK=30), max_batch=5, max_vocab=999)
    t.SetConfig(rocm.SamplerConfig(TopK=30, FrequencyPenalty=0.7))
    got = rocm.sample_host(t, x, u, hist)
    fx = oracle.sample(x, u, 1.0, 30, 1.0, 1.0, hist, mode=oracle.MODE_FIXED, freq=0.7)
    assert np.array_equal(got["tokens"], fx["tokens"])
    t.SetConfig(rocm.SamplerConfig(TopK=30))
    got = rocm.sample_host(t, x, u, hist)
    fx = oracle.sample(x, u, 1.0, 30, 1.0, 1.0, hist, mode=oracle.MODE_FIXED)
    assert np.array_equal(got["tokens"], fx["tokens"])
    # no history: the penalties have nothing to act on
    got = rocm.sample_host(s, x, u, None)
    fx = oracle.sample(x, u, 1.0, 30, 0.9, 1.1, None, mode=oracle.MODE_FIXED)
    assert np.array_equal(got["tokens"], fx["tokens"])
    for h in (s, t):
        h.Status()
        h.Close()


@pytest.mark.parametrize("H", [400, 3000, 4096, 5000])
def test_frequency_penalty_rows_the_single_pass_kernel_cannot_prove(oracle, rocm, H):
    # fewer finite logits than top_k, and heavy ties: the workgroup finishes by its exact selection, which penalises
    # every element it ranks (occurrences counted in its own hash of the history up to 4096 tokens, read from the
    # handle's table beyond)
    rng = np.random.default_rng(78 + H)
    B, V = 8, 5000
    x = np.full((B, V), -np.inf, dtype=np.float32)
    x[:, :30] = rng.standard_normal((B, 30), dtype=np.float32)
    x[4:] = np.float32(1.0)                                                # every logit ties
    u = rng.random(B, dtype=np.float32)
    hist = rng.integers(0, 40, size=(B, H)).astype(np.int32)
    hist[1::2] = rng.integers(0, V, size=(B // 2, H)).astype(np.int32)    # many distinct ids in every other row
    got, _, _ = _check_against_oracle(oracle, rocm, x, u, 0.8, 50, 0.95, 1.2, hist, nuc=50, freq=0.01, pres=0.02)
    assert got["counters"]["fallback_rows"] > 0


def test_frequency_and_presence_penalties_are_validated(rocm):
    for kw in (dict(FrequencyPenalty=float("inf")), dict(PresencePenalty=float("nan"))):
        with pytest.raises(rocm.SamplerPanic, match="penalty"):
            rocm.NewSampler(rocm.SamplerConfig(**kw), max_batch=1, max_vocab=16)
    s = rocm.NewSampler(rocm.SamplerConfig(FrequencyPenalty=-0.5, PresencePenalty=0.25), max_batch=1, max_vocab=16)
    c = s.Config()
    assert c.FrequencyPenalty == -0.5 and c.PresencePenalty == 0.25
    s.Close()


# ---------------------------------------------------------------- token log-probabilities and cross-entropy
# A floating-point quantity (one sweep, online log-sum-exp): within 1e-5 + 1e-6 |value| of the fp64 truth (and of the
# oracle's integer-normaliser form, which is that close to the truth itself), and within 1e-4 * max(1, |x|max * 1e-2) + V * 2^-25 of the reference's fp32 arithmetic (whose sequential fp32 sum of V terms
# is the less accurate side).

@pytest.mark.parametrize("B,V,T,rep,H,freq,pres", [
    (32, 128256, 0.7, 1.15, 512, 0.0, 0.0),       # C3 shape
    (32, 128256, 1.0, 1.0, 0, 0.0, 0.0),          # plain log-softmax gather: the cross-entropy term
    (16, 152064, 1.2, 1.05, 2048, 0.2, 0.3),      # C5 shape with every penalty
    (9, 1001, 0.5, 0.8, 300, -0.1, 0.4),          # unaligned rows, boosting penalties
    (5, 3, 1.0, 1.0, 0, 0.0, 0.0),
    (5, 1, 2.0, 1.0, 0, 0.0, 0.0),
    (4096, 10, 1.0, 1.0, 0, 0.0, 0.0),            # short rows without a history: a group of lanes per row (4, 16 or 64 by length)
    (300, 100, 0.7, 1.0, 0, 0.0, 0.0),
    (70, 4096, 1.3, 1.0, 0, 0.0, 0.0),
    (9, 4095, 1.0, 1.0, 0, 0.0, 0.0),
    (33, 17, 2.0, 1.0, 0, 0.0, 0.0),
    (300, 8193, 1.0, 1.0, 0, 0.0, 0.0),           # more rows than CUs: the 512-thread instance by the default selection
    (520, 5000, 0.8, 1.2, 100, 0.1, 0.0),
])
@pytest.mark.parametrize("path", [0, 2])          # 2: the 512-thread instance (two rows to a CU) whatever the batch
def test_token_logprobs_against_oracle(oracle, rocm, B, V, T, rep, H, freq, pres, path):
    rng = np.random.default_rng(B * 31 + V)
    x = (rng.standard_normal((B, V), dtype=np.float32) * np.float32(2.5)).astype(np.float32)
    tok = rng.integers(0, V, B).astype(np.int32)
    tok[0] = int(np.argmax(x[0]))
    hist = ((rng.zipf(1.2, size=(B, H)) - 1) % V).astype(np.int32) if H else None
    if H:
        tok[1:4] = hist[1:4, 0]                                            # penalised tokens among the queried ones
    hist_len = rng.integers(H // 2, H + 1, size=B).astype(np.int32) if H else None
    s = rocm.NewSampler(rocm.SamplerConfig(Temperature=T, RepetitionPenalty=rep, FrequencyPenalty=freq, PresencePenalty=pres,
                                           TopK=5, TopP=0.5, MinP=0.1),     # truncation settings do not enter
                        max_batch=B, max_vocab=V)
    s.SetPath(path)
    got = rocm.token_logprobs_host(s, x, tok, hist, hist_len)
    s.Status()
    s.Close()
    kw = dict(temperature=T, rep=rep, history=hist, hist_len=hist_len, freq=freq, pres=pres)
    fx, _ = oracle.token_logprobs(x, tok, mode=oracle.MODE_FIXED, **kw)
    tr, _ = oracle.token_logprobs(x, tok, mode=oracle.MODE_TRUTH, **kw)
    rf, _ = oracle.token_logprobs(x, tok, mode=oracle.MODE_REF32, **kw)
    assert np.all(np.abs(got.astype(np.float64) - tr) <= 1e-5 + 1e-6 * np.abs(tr))
    assert np.all(np.abs(got.astype(np.float64) - fx) <= 1e-5 + 1e-6 * np.abs(fx))
    # the reference sums the V exponentials sequentially in fp32: its own rounding, up to V * 2^-24 relative in the
    # normaliser, is what separates it from the truth at large V
    assert np.max(np.abs(got - rf)) <= 1e-4 * max(1.0, float(np.abs(x).max()) / T * 1e-2) + V * 2.0 ** -25
    assert (got <= 0).all()


def test_token_logprobs_match_the_sampler_and_special_rows(oracle, rocm):
    rng = np.random.default_rng(5)
    B, V, H = 24, 32000, 64
    x = (rng.standard_normal((B, V), dtype=np.float32) * np.float32(2.0)).astype(np.float32)
    u = rng.random(B, dtype=np.float32)
    hist = ((rng.zipf(1.2, size=(B, H)) - 1) % V).astype(np.int32)
    s = rocm.NewSampler(rocm.SamplerConfig(Temperature=0.8, RepetitionPenalty=1.2, PresencePenalty=0.3), max_batch=B, max_vocab=V)
    smp = rocm.sample_host(s, x, u, hist)                                   # no truncation: probs are the full softmax's
    lp = rocm.token_logprobs_host(s, x, smp["tokens"], hist)
    assert np.allclose(np.exp(lp.astype(np.float64)), smp["probs"], rtol=1e-5)
    # nothing finite: every token ties; a masked token: -inf; a token outside the vocabulary: NaN and a data error
    y = np.full((3, 1000), -np.inf, dtype=np.float32)
    y[1, 2] = 0.0
    y[2, :] = 1.0
    lp = rocm.token_logprobs_host(s, y, np.array([3, 5, 999], np.int32))
    s.Status()
    assert abs(lp[0] + np.log(1000.0)) < 1e-6 and lp[1] == -np.inf and abs(lp[2] + np.log(1000.0)) < 1e-6
    lp = rocm.token_logprobs_host(s, y, np.array([0, 2, 1000], np.int32))
    assert lp[1] == 0.0 and np.isnan(lp[2])
    with pytest.raises(rocm.BornRocmError):
        s.Status()
    s.Status()
    with pytest.raises(rocm.SamplerPanic, match="null tokens"):
        s.TokenLogprobs(rocm.DeviceBuffer(16), 1, 4, None, None, None, rocm.DeviceBuffer(4))
    s.Close()


def test_cross_entropy_loss_mirror(oracle, rocm):
    import json
    import os
    from born_amd.loss import CrossEntropyLoss
    from test_oracle_reference_kats import check_cross_entropy_case
    with open(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "reference_kats.json")) as f:
        kats = json.load(f)["cross_entropy"]
    crit = CrossEntropyLoss(max_batch=64, max_vocab=50000)

    def loss_of(x, t):
        return crit.Forward(rocm.DeviceBuffer.from_numpy(x), x.shape, rocm.DeviceBuffer.from_numpy(t))

    for case in kats:                                                       # what the reference's own tests assert
        check_cross_entropy_case(case, loss_of)
    rng = np.random.default_rng(6)
    for (B, V) in [(64, 50000), (7, 10), (1, 32000)]:
        x = (rng.standard_normal((B, V)) * 3.0).astype(np.float32)
        t = rng.integers(0, V, B).astype(np.int32)
        got = loss_of(x, t)
        assert got.dtype == np.float32
        assert abs(float(got) - oracle.cross_entropy_ref(x, t)) <= 1e-5 * max(1.0, abs(float(got)))
    with pytest.raises(rocm.SamplerPanic, match="logits must be 2D"):
        crit.Forward(rocm.DeviceBuffer(16), (4,), rocm.DeviceBuffer(16))
    with pytest.raises(rocm.SamplerPanic, match="targets must have shape"):
        crit.Forward(rocm.DeviceBuffer(32), (2, 4), rocm.DeviceBuffer(12))
    assert crit.Parameters() == []
    crit.Close()


# path 2: the three-sweep kernel with 512 threads per row (what batches of more rows than CUs get), path 0: 1024
NUCLEUS_PATHS = [0, 2]


@pytest.mark.parametrize("path", NUCLEUS_PATHS)
@pytest.mark.parametrize("V,pad", [(7, 5), (7, 1), (6, 2), (4102, 2), (4103, 1), (8198, 2)])
def test_three_sweep_kernel_ragged_tail_after_a_partial_wave(oracle, rocm, V, pad, path):
    # 16-byte aligned rows whose length is not a multiple of four, with the whole float4 blocks ending at lane 0 or 1 of a
    # wave: the ragged tail restarts at lane 0, next to lanes that sat out the last block.  Few distinct values, so that
    # the wanted bins take entries from both parts.
    rng = np.random.default_rng(V * 31 + pad)
    B, H = 6, 40
    x = np.round(rng.standard_normal((B, V)) * 0.6).astype(np.float32)
    x[0, :] = np.float32(0.25)
    u = rng.random(B, dtype=np.float32)
    hist = rng.integers(0, V, size=(B, H)).astype(np.int32)
    stride = V + pad
    assert stride % 4 == 0
    host = np.full(B * stride + 8, np.nan, dtype=np.float32)
    for b in range(B):
        host[b * stride: b * stride + V] = x[b]
    for (T, p, rep, min_p, freq) in [(5.0, 0.9, 1.0, 0.05, 0.1), (1.0, 0.9, 1.2, 0.0, 0.0), (0.7, 1.0, 1.0, 0.0, 0.0)]:
        s = rocm.NewSampler(rocm.SamplerConfig(Temperature=T, TopK=0, TopP=p, RepetitionPenalty=rep, MinP=min_p, FrequencyPenalty=freq),
                            max_batch=B, max_vocab=V)
        s.SetPath(path)
        d_x, d_u, d_h = rocm.DeviceBuffer.from_numpy(host), rocm.DeviceBuffer.from_numpy(u), rocm.DeviceBuffer.from_numpy(hist)
        tok, pr = rocm.DeviceBuffer(4 * B), rocm.DeviceBuffer(4 * B)
        s.Sample(d_x, B, V, d_h, None, d_u, tok, pr, row_stride=stride, hist_stride=H)
        s.Status()
        fx = oracle.sample(x, u, T, 0, p, rep, hist, None, mode=oracle.MODE_FIXED, min_p=min_p, freq=freq)
        assert np.array_equal(tok.to_numpy(np.int32, (B,)), fx["tokens"]), (T, p, rep, min_p, freq)
        assert np.array_equal(pr.to_numpy(np.float32, (B,)).view(np.uint32), fx["probs"].view(np.uint32))
        assert s.Counters()["general_rows"] == B
        s.Close()


@pytest.mark.parametrize("path", NUCLEUS_PATHS)
@pytest.mark.parametrize("pad_extra", [0, 4])
def test_three_sweep_kernel_every_row_length_residue(oracle, rocm, pad_extra, path):
    # every vocabulary size modulo 256 (so: every way the row's last whole 128-bit blocks and its ragged tail can fall
    # on the lanes of a wave), at two row pitches; few distinct values, so that the wanted bins take entries from all
    # parts of the row and a lost or duplicated staged entry changes the result
    B, H = 3, 24
    for V in range(4096, 4096 + 256):
        rng = np.random.default_rng(V * 7 + pad_extra)
        x = np.round(rng.standard_normal((B, V)) * 0.6).astype(np.float32)
        u = rng.random(B, dtype=np.float32)
        hist = rng.integers(0, V, size=(B, H)).astype(np.int32)
        stride = ((V + 3) & ~3) + pad_extra
        host = np.full(B * stride + 8, np.nan, dtype=np.float32)
        for b in range(B):
            host[b * stride: b * stride + V] = x[b]
        T, p, rep = (1.0, 0.9, 1.2) if V % 2 else (0.7, 1.0, 1.0)
        s = rocm.NewSampler(rocm.SamplerConfig(Temperature=T, TopK=0, TopP=p, RepetitionPenalty=rep), max_batch=B, max_vocab=V)
        s.SetPath(path)
        d_x, d_u, d_h = rocm.DeviceBuffer.from_numpy(host), rocm.DeviceBuffer.from_numpy(u), rocm.DeviceBuffer.from_numpy(hist)
        tok, pr = rocm.DeviceBuffer(4 * B), rocm.DeviceBuffer(4 * B)
        s.Sample(d_x, B, V, d_h, None, d_u, tok, pr, row_stride=stride, hist_stride=H)
        s.Status()
        fx = oracle.sample(x, u, T, 0, p, rep, hist, None, mode=oracle.MODE_FIXED)
        assert np.array_equal(tok.to_numpy(np.int32, (B,)), fx["tokens"]), (V, pad_extra)
        assert np.array_equal(pr.to_numpy(np.float32, (B,)).view(np.uint32), fx["probs"].view(np.uint32)), (V, pad_extra)
        s.Close()


@pytest.mark.parametrize("path", NUCLEUS_PATHS)
@pytest.mark.parametrize("T", [0.7, 1.2, 0.35, 1.9999999, 1.0])
def test_three_sweep_kernel_division_shortcut_and_unusual_magnitudes(oracle, rocm, T, path):
    """Without a top-k cut every logit is divided by the temperature. For most temperatures the kernel replaces the
    division by a multiplication and two fused multiply-adds that give the same quotient for logits of ordinary
    magnitude (1.9999999 is a temperature it must divide by); zeros, denormals, tiny and huge values, infinities
    and NaNs take the division itself. All of them, mixed into ordinary rows: bit-exact against the oracle."""
    rng = np.random.default_rng(int(T * 1e6))
    B, V = 12, 20011
    x = (rng.standard_normal((B, V)) * 2.5).astype(np.float32)
    odd = np.array([0.0, -0.0, 1e-45, -1e-45, 1e-39, 3e-31, -3e-31, 7.9e-31, 2 ** -100, -(2 ** -100), 2 ** -101, 1.2e30, -1.2e30,
                    2 ** 100, 2 ** 99, -(2 ** 100), 3e38, -3e38, np.inf, -np.inf, np.nan], dtype=np.float32)
    # values that leave the row's maximum ordinary (such rows take the sweeps that test no logit's magnitude)
    low = np.array([0.0, -0.0, 1e-45, -1e-45, 1e-39, 3e-31, -3e-31, 7.9e-31, 2 ** -100, -(2 ** -100), 2 ** -101, -1.2e30,
                    -(2 ** 100), -(2 ** 99), -3e38, -np.inf, np.nan], dtype=np.float32)
    for b in range(1, B):
        at = rng.choice(V, size=40 * b, replace=False)
        # (rows b % 3 == 0: no infinities, no huge values; b % 3 == 1: nothing above the ordinary maximum)
        x[b, at] = rng.choice(odd[:17] if b % 3 == 0 else low if b % 3 == 1 else odd, size=at.size)
    x[5, :] = rng.choice(np.array([0.0, -0.0, 1e-45, 2 ** -101, 3e-31], dtype=np.float32), size=V)   # nothing of ordinary magnitude
    u = rng.random(B, dtype=np.float32)
    hist = rng.integers(0, V, size=(B, 64)).astype(np.int32)
    for p, rep, min_p in [(0.9, 1.0, 0.0), (1.0, 1.3, 0.0), (0.97, 1.1, 0.02)]:
        got, _, _ = _check_against_oracle(oracle, rocm, x, u, T, 0, p, rep, hist if rep != 1.0 else None, min_p=min_p, path=path)
        assert got["counters"]["general_rows"] == B and got["counters"]["topk_rows"] == 0


@pytest.mark.parametrize("path", NUCLEUS_PATHS)
@pytest.mark.parametrize("V,H,scale", [(50, 40, 1.0), (300, 900, 1.0), (5000, 2048, 1.0), (6000, 2100, 1.0), (6000, 4200, 1.0),
                                       (5000, 600, 3e6), (4099, 4096, 1.0)])
def test_three_sweep_kernel_seen_ids_visited_apart(oracle, rocm, V, H, scale, path):
    """With penalties on, the kernel lists the ids of the history once each, keeps their penalised logits in registers
    (up to four per thread: 2048 ids at 512 threads per row, 4096 at 1024) and shows the sweeps a constant in their
    place; longer histories, and rows whose maximum is too large for such a constant, keep the penalty inside the
    sweeps. Both ways, with repeated ids, with draws from the very end of the rank order (where the constant's own
    bin is the wanted one) and with the counted penalties: bit-exact against the oracle."""
    rng = np.random.default_rng(V * 13 + H)
    B = 8
    x = (rng.standard_normal((B, V)) * scale).astype(np.float32)
    hist = ((rng.zipf(1.3, size=(B, H)) - 1) % V).astype(np.int32)
    hist[:, ::3] = rng.integers(0, V, size=hist[:, ::3].shape)
    hl = rng.integers(max(1, H - 3), H + 1, size=B).astype(np.int32)
    u = rng.random(B, dtype=np.float32)
    u[0] = np.float32(1.0) - np.float32(2.0 ** -24)        # the last element in rank order
    u[1] = np.float32(0.99999)
    u[2] = 0.0
    for (T, p, rep, freq, pres) in [(3.0, 1.0, 1.3, 0.0, 0.0), (1.2, 0.999, 1.05, 0.0, 0.0), (2.0, 1.0, 1.0, 0.3, 0.2),
                                    (0.8, 0.9, 2.0, 0.1, 0.0)]:
        got, _, _ = _check_against_oracle(oracle, rocm, x, u, T * scale, 0, p, rep, hist, hl, path=path, freq=freq, pres=pres)
        assert got["counters"]["general_rows"] == B


@pytest.mark.parametrize("path", NUCLEUS_PATHS)
@pytest.mark.parametrize("T,V", [(1.0, 9001), (0.8, 9001), (1.9999999, 9001), (0.8, 40003), (1.0, 70000)])
def test_three_sweep_kernel_seen_logits_above_the_penalised_maximum(oracle, rocm, T, V, path):
    """Rows whose largest stored logits belong to ids of the history, far above everything else, so that after the
    penalty the maximum is another logit or a much smaller value: the sweeps that read the logits as stored meet
    values above the maximum they work from, up to overflow of the exponential, and what they add for them must
    come out again exactly; and the first sweep, which keeps a maximum per stage of the row and reads again the
    stages whose maximum a seen id holds, reads several of them again. Also with unusual values among the seen ids.
    Bit-exact against the oracle."""
    rng = np.random.default_rng(int(T * 1000) + 5 + V)
    B, H = 10, 200
    x = rng.standard_normal((B, V)).astype(np.float32)
    hist = rng.integers(0, V, size=(B, H)).astype(np.int32)
    tops = [60.0, 25.0, 300.0, 3000.0, 1e9, 12.0, 88.5, 1e30, 40.0, 14.0]
    for b in range(B):
        x[b, hist[b, :3 + b % 4]] = np.float32(tops[b]) * (1 + 0.01 * np.arange(3 + b % 4, dtype=np.float32))
        x[b, hist[b, 10:20]] = np.array([0.0, -0.0, 1e-45, -np.inf, np.nan, -3e38, 2 ** -101, -1e-39, 5.0, -5.0], dtype=np.float32)
    u = rng.random(B, dtype=np.float32)
    for p, rep, freq, pres in [(0.95, 10.0, 0.0, 0.0), (1.0, 1.3, 0.0, 0.0), (0.9, 100.0, 0.0, 0.0), (0.99, 1.0, 2.0, 30.0)]:
        got, _, _ = _check_against_oracle(oracle, rocm, x, u, T, 0, p, rep, hist, path=path, freq=freq, pres=pres)
        assert got["counters"]["general_rows"] == B


@pytest.mark.parametrize("path", NUCLEUS_PATHS)
@pytest.mark.parametrize("V,peaks,lift", [(4096, 3, 14.0), (32000, 20, 9.0), (50000, 200, 6.0), (128256, 20, 9.0), (20000, 700, 7.0)])
def test_three_sweep_kernel_peaked_rows_gather_the_nucleus_whole(oracle, rocm, V, peaks, lift, path):
    """Top-p alone on peaked rows (what a trained model emits): a few lifted logits carry nearly all of the mass, the
    cut's bin holds so much of it that the draw may fall into any of many bins, all of which the kernel gathers with the
    cut's. From a handful of peaks to more than the lists hold (the row then takes the radix descent), with and without penalties on the peaks
    themselves: bit-exact against the oracle."""
    rng = np.random.default_rng(V + peaks)
    B = 12
    x = (rng.standard_normal((B, V)) * 1.5).astype(np.float32)
    hist = rng.integers(0, V, size=(B, 64)).astype(np.int32)
    for b in range(B):
        at = rng.choice(V, size=peaks, replace=False)
        x[b, at] += rng.uniform(lift * 0.6, lift * 1.3, size=peaks).astype(np.float32)
        hist[b, :8] = at[:8] if peaks >= 8 else np.resize(at, 8)     # some of the peaks are penalised
    x[1, :] = x[1, 0]                                                  # a flat row among them
    x[2, rng.choice(V, size=2, replace=False)] = 40.0                  # two equal maxima far above the rest
    hl = np.full(B, hist.shape[1], dtype=np.int32)
    u = rng.random(B, dtype=np.float32)
    u[0] = np.float32(1.0) - np.float32(2.0 ** -24)
    u[3] = 0.0
    for (T, p, rep) in [(0.7, 0.9, 1.15), (1.0, 0.5, 1.0), (1.0, 0.99, 1.3), (1.4, 0.999, 1.0), (0.5, 0.2, 2.0)]:
        got, _, _ = _check_against_oracle(oracle, rocm, x, u, T, 0, p, rep, hist, hl, path=path)
        assert got["counters"]["general_rows"] == B


def test_three_sweep_kernel_random_case_that_lost_staged_entries(oracle, rocm):
    # the case a wide seeded sweep of test_random_row_layouts_against_oracle found (its chunk 1096, third case)
    import test_gpu_parity_random as R
    rng = np.random.default_rng(777 + 1096)
    for _ in range(3):
        c = R._draw_case(rng)
        x, u, hist, hist_len = R._inputs(rng, c)
        rng.choice([0, 1, 3, 4, 5, 64]), rng.choice([0, 1, 2, 3, 4])     # that test's padding and offset draws
    assert c["V"] == 7 and c["k"] >= c["V"]
    B, V = x.shape
    stride = V + 5
    host = np.full(B * stride + 8, np.nan, dtype=np.float32)
    host[1::2] = np.inf
    for b in range(B):
        host[b * stride: b * stride + V] = x[b]
    s = rocm.NewSampler(rocm.SamplerConfig(Temperature=c["T"], TopK=c["k"], TopP=c["p"], RepetitionPenalty=c["rep"], MinP=c["min_p"],
                                           FrequencyPenalty=c["freq"], PresencePenalty=c["pres"]), max_batch=B, max_vocab=V)
    d_x, d_u, d_h = rocm.DeviceBuffer.from_numpy(host), rocm.DeviceBuffer.from_numpy(u), rocm.DeviceBuffer.from_numpy(hist)
    tok = rocm.DeviceBuffer(4 * B)
    s.Sample(d_x, B, V, d_h, None, d_u, tok, None, row_stride=stride, hist_stride=hist.shape[1])
    s.Status()
    fx = oracle.sample(x, u, c["T"], c["k"], c["p"], c["rep"], hist, hist_len, mode=oracle.MODE_FIXED, min_p=c["min_p"], freq=c["freq"],
                       pres=c["pres"])
    assert np.array_equal(tok.to_numpy(np.int32, (B,)), fx["tokens"])
    s.Close()


@pytest.mark.parametrize("path", NUCLEUS_PATHS)
@pytest.mark.parametrize("V", [8, 64, 100, 130, 4100])
def test_three_sweep_kernel_rows_that_end_inside_a_wave(oracle, rocm, V, path):
    # no top-k cut and a row whose last elements occupy only part of a wave: the lanes that sit out the ragged end
    # must still see every entry the wave gathered (heavy ties make the gathered bins full)
    rng = np.random.default_rng(V)
    x = np.round(rng.standard_normal((6, V))).astype(np.float32)
    u = rng.random(6, dtype=np.float32)
    for p in (1.0, 0.9):
        _check_against_oracle(oracle, rocm, x, u, T=5.0, k=0, p=p, path=path)


def test_builtin_uniform_stream_in_sample(oracle, rocm):
    rng = np.random.default_rng(9)
    B, V = 16, 6000
    x = rng.standard_normal((B, V), dtype=np.float32)
    s = rocm.NewSampler(rocm.SamplerConfig(TopK=30, Seed=4242), max_batch=B, max_vocab=V)
    for step in range(3):
        got = rocm.sample_host(s, x, None)
        u = np.array([oracle.uniform(4242, step, r) for r in range(B)], dtype=np.float32)
        want = oracle.sample(x, u, top_k=30, mode=oracle.MODE_FIXED)
        assert np.array_equal(got["tokens"], want["tokens"]), step


# ---------------------------------------------------------------- speculative accept / reject

def test_spec_verify_against_oracle(oracle, rocm):
    from born_amd import synth
    w = synth.c4(rows=16)
    e = w.extra
    s = rocm.NewSampler(max_batch=16, max_vocab=32000)
    got = rocm.verify_host(s, e["target"], e["draft"], e["draft_tokens"], e["u_acc"], e["u_res"])
    fx = oracle.spec_verify(e["target"], e["draft"], e["draft_tokens"], e["u_acc"], e["u_res"], mode=oracle.MODE_FIXED)
    tr = oracle.spec_verify(e["target"], e["draft"], e["draft_tokens"], e["u_acc"], e["u_res"], mode=oracle.MODE_TRUTH)
    assert np.array_equal(got["n_accepted"], fx["n_accepted"]) and np.array_equal(got["next_token"], fx["next_token"])
    diff = (got["n_accepted"] != tr["n_accepted"]) | (got["next_token"] != tr["next_token"])
    assert not (diff & ~tr["near"]).any()
    assert 0 < got["n_accepted"].mean() < 5                               # the workload exercises both outcomes
    s.Status()


def test_spec_verify_special_cases(oracle, rocm):
    rng = np.random.default_rng(10)
    B, G, V = 6, 5, 3001                                                   # odd vocabulary: scalar load path
    t = rng.standard_normal((B, G, V), dtype=np.float32)
    d = rng.integers(0, V, size=(B, G)).astype(np.int32)
    ua, ur = rng.random((B, G), dtype=np.float32), rng.random(B, dtype=np.float32)
    s = rocm.NewSampler(rocm.SamplerConfig(Temperature=0.8), max_batch=B, max_vocab=V)
    got = rocm.verify_host(s, t, t.copy(), d, ua, ur)                      # identical models accept everything
    assert np.all(got["n_accepted"] == G) and np.all(got["next_token"] == -1)
    dr = (t + rng.standard_normal((B, G, V), dtype=np.float32)).astype(np.float32)
    got = rocm.verify_host(s, t, dr, d, ua, ur)
    fx = oracle.spec_verify(t, dr, d, ua, ur, temperature=0.8, mode=oracle.MODE_FIXED)
    assert np.array_equal(got["n_accepted"], fx["n_accepted"]) and np.array_equal(got["next_token"], fx["next_token"])
    # hand vector: p = [.5 .3 .2], q = [.2 .5 .3], draft token 1 -> accept iff u < 0.6, residual -> id 0
    s1 = rocm.NewSampler(max_batch=1, max_vocab=3)
    tt = np.log(np.array([[[5, 3, 2]]], dtype=np.float64)).astype(np.float32)
    qq = np.log(np.array([[[2, 5, 3]]], dtype=np.float64)).astype(np.float32)
    r = rocm.verify_host(s1, tt, qq, np.array([[1]], np.int32), np.array([[0.59]], np.float32), np.array([0.7], np.float32))
    assert r["n_accepted"][0] == 1 and r["next_token"][0] == -1
    r = rocm.verify_host(s1, tt, qq, np.array([[1]], np.int32), np.array([[0.61]], np.float32), np.array([0.7], np.float32))
    assert r["n_accepted"][0] == 0 and r["next_token"][0] == 0
    # out-of-range draft token: rejected, reported through the status word
    bad = d.copy()
    bad[2, 0] = V + 5
    got = rocm.verify_host(s, t, dr, bad, ua, ur)
    assert got["n_accepted"][2] == 0
    with pytest.raises(rocm.BornRocmError):
        s.Status()
    s.Status()                                                             # the status word clears once read


@pytest.mark.parametrize("T", [1.0, 0.8, 1.9999999])
@pytest.mark.parametrize("V", [32000, 3001, 40000])
def test_spec_verify_unusual_logits(oracle, rocm, T, V):
    """Zeros of both signs, denormals, tiny and hugely negative values, -inf (masked tokens) and NaNs mixed into both
    models' rows under maxima of ordinary size (the kernels then compute every mass without a test of the logit), rows
    with +inf or huge maxima (which take the tested arithmetic), and a draft that masks what the target prefers:
    accept counts and tokens bit-exact against the oracle, resident, scalar and two-sweep rows, with and without the
    division shortcut (1.9999999 has none)."""
    rng = np.random.default_rng(V + int(T * 100))
    B, G = 8, 3
    t = (rng.standard_normal((B, G + 1, V)) * 2).astype(np.float32)
    dr = (t[:, :G] + 0.7 * rng.standard_normal((B, G, V))).astype(np.float32)
    low = np.array([0.0, -0.0, 1e-45, -1e-45, 1e-39, 3e-31, -3e-31, 2 ** -100, -(2 ** -100), 2 ** -101, -1.2e30, -(2 ** 100),
                    -3e38, -np.inf, np.nan], dtype=np.float32)
    for b in range(B):
        for g in range(G + 1):
            at = rng.choice(V, size=50 + 10 * b, replace=False)
            t[b, g, at] = rng.choice(low, size=at.size)
            if g < G:
                at = rng.choice(V, size=50 + 10 * b, replace=False)
                dr[b, g, at] = rng.choice(low, size=at.size)
    t[6, 1, 17] = np.inf                                                  # rows outside the usual kind
    dr[6, 2, 5] = 3e38
    t[7, 0, 99] = 2.0 ** 101
    dr[5, 0, np.argsort(t[5, 0])[-40:]] = -np.inf                          # the draft masks the target's favourites
    d = rng.integers(0, V, size=(B, G)).astype(np.int32)
    ua, ur = rng.random((B, G), dtype=np.float32), rng.random(B, dtype=np.float32)
    s = rocm.NewSampler(rocm.SamplerConfig(Temperature=T), max_batch=B, max_vocab=V)
    got = rocm.verify_host(s, t, dr, d, ua, ur, bonus=True)
    tt, bonus = np.ascontiguousarray(t[:, :G]), np.ascontiguousarray(t[:, G])
    fx = oracle.spec_verify(tt, dr, d, ua, ur, temperature=T, mode=oracle.MODE_FIXED, bonus=bonus)
    assert np.array_equal(got["n_accepted"], fx["n_accepted"]), (T, V)
    assert np.array_equal(got["next_token"], fx["next_token"]), (T, V)
    s.Status()
    s.Close()


def test_spec_verify_bonus_draw(oracle, rocm):
    # target given as [B, G + 1, V] (the bonus row is the last position, addressed through sequence strides)
    rng = np.random.default_rng(31)
    for (B, G, V, T) in [(24, 4, 32000, 1.0), (7, 3, 3001, 0.8), (3, 2, 40000, 1.3)]:   # resident / scalar / two-sweep rows
        t = rng.standard_normal((B, G + 1, V), dtype=np.float32)
        dr = t[:, :G].copy()
        half = B // 2
        dr[half:] += (0.6 * rng.standard_normal((B - half, G, V))).astype(np.float32)   # first half: identical models
        d = rng.integers(0, V, size=(B, G)).astype(np.int32)
        ua, ur = rng.random((B, G), dtype=np.float32), rng.random(B, dtype=np.float32)
        s = rocm.NewSampler(rocm.SamplerConfig(Temperature=T), max_batch=B, max_vocab=V)
        got = rocm.verify_host(s, t, dr, d, ua, ur, bonus=True)
        tt, bonus = np.ascontiguousarray(t[:, :G]), np.ascontiguousarray(t[:, G])
        fx = oracle.spec_verify(tt, dr, d, ua, ur, temperature=T, mode=oracle.MODE_FIXED, bonus=bonus)
        tr = oracle.spec_verify(tt, dr, d, ua, ur, temperature=T, mode=oracle.MODE_TRUTH, bonus=bonus)
        assert np.array_equal(got["n_accepted"], fx["n_accepted"]), (B, G, V)
        assert np.array_equal(got["next_token"], fx["next_token"]), (B, G, V)
        diff = (got["n_accepted"] != tr["n_accepted"]) | (got["next_token"] != tr["next_token"])
        assert not (diff & ~tr["near"]).any()
        assert np.all(got["n_accepted"][:half] == G) and np.all(got["next_token"] >= 0)
        # without bonus rows the same call leaves -1 for the fully accepted sequences
        plain = rocm.verify_host(s, tt, dr, d, ua, ur)
        assert np.array_equal(plain["n_accepted"], got["n_accepted"])
        assert np.all(plain["next_token"][:half] == -1)
        rej = got["n_accepted"] < G
        assert np.array_equal(plain["next_token"][rej], got["next_token"][rej])
        s.Status()
        s.Close()
    # uniform bonus row: token = floor(u V)
    B, G, V = 4, 1, 1000
    t = np.zeros((B, G + 1, V), np.float32)
    t[:, 0] = rng.standard_normal((B, V), dtype=np.float32)
    ur = np.array([0.0, 0.4995, 0.5005, 0.9999], np.float32)
    s = rocm.NewSampler(max_batch=B, max_vocab=V)
    got = rocm.verify_host(s, t, t[:, :1].copy(), np.zeros((B, 1), np.int32), np.full((B, 1), 0.5, np.float32), ur, bonus=True)
    assert got["next_token"].tolist() == [0, 499, 500, 999]


# ---------------------------------------------------------------- a configuration per row

def _sample_rows(rocm, x, u, hist, Ts, ks, ps, reps, path=0, min_ps=None, freqs=None, press=None, row_kinds=0, **handle):
    B, V = x.shape
    s = rocm.NewSampler(rocm.SamplerConfig(Temperature=0.9, TopK=7, TopP=0.8, RepetitionPenalty=1.3, **handle), max_batch=B, max_vocab=V)
    s.SetPath(path)
    dev = lambda a, dt: None if a is None else rocm.DeviceBuffer.from_numpy(np.ascontiguousarray(a, dtype=dt))
    tok, pr = rocm.DeviceBuffer(4 * B), rocm.DeviceBuffer(4 * B)
    s.SampleRows(dev(x, np.float32), B, V, dev(hist, np.int32), None, dev(u, np.float32), dev(Ts, np.float32), dev(ks, np.int32),
                 dev(ps, np.float32), dev(reps, np.float32), tok, pr, hist_stride=0 if hist is None else hist.shape[1],
                 minPs=dev(min_ps, np.float32), frequencyPenalties=dev(freqs, np.float32), presencePenalties=dev(press, np.float32),
                 rowKinds=row_kinds)
    return s, tok.to_numpy(np.int32, (B,)), pr.to_numpy(np.float32, (B,))


@pytest.mark.parametrize("path", [0, 1, 2])
def test_per_row_configurations_match_per_row_handles(oracle, rocm, path):
    # one batch, every row its own settings, covering the three kernels' territories (top-k <= 512, no top-k cut,
    # top-k > 64, a boosting penalty < 1); each row must equal the oracle under that row's settings
    rng = np.random.default_rng(77)
    B, V, H = 24, 9000, 48
    x = (rng.standard_normal((B, V)) * 2.0).astype(np.float32)
    u = rng.random(B, dtype=np.float32)
    hist = rng.integers(0, V, (B, H)).astype(np.int32)
    Ts = rng.choice([0.5, 0.7, 1.0, 1.3], B).astype(np.float32)
    ks = rng.choice([0, 1, 5, 40, 64, 65, 128, 300, 512, 513, 900, V, V + 5, -3], B).astype(np.int32)
    ps = rng.choice([1.0, 0.9, 0.5, 0.99], B).astype(np.float32)
    reps = rng.choice([1.0, 1.15, 2.0, 0.8], B).astype(np.float32)
    s, tok, pr = _sample_rows(rocm, x, u, hist, Ts, ks, ps, reps, path)
    s.Status()
    for b in range(B):
        want = oracle.sample(x[b:b + 1], u[b:b + 1], float(Ts[b]), int(ks[b]), float(ps[b]), float(reps[b]), hist[b:b + 1], None,
                             mode=oracle.MODE_FIXED)
        assert tok[b] == want["tokens"][0], (b, Ts[b], ks[b], ps[b], reps[b])
        assert pr[b:b + 1].view(np.uint32)[0] == want["probs"].view(np.uint32)[0], b
    # arrays left out fall back to the handle's values (T 0.9, top_k 7, top_p 0.8, penalty 1.3)
    s2, tok2, pr2 = _sample_rows(rocm, x, u, hist, None, ks, None, None, path)
    s2.Status()
    for b in range(B):
        want = oracle.sample(x[b:b + 1], u[b:b + 1], 0.9, int(ks[b]), 0.8, 1.3, hist[b:b + 1], None, mode=oracle.MODE_FIXED)
        assert tok2[b] == want["tokens"][0], b
    if path != 1:
        c = s.Counters()
        assert c["topk_rows"] > 0 and c["general_rows"] > 0                 # more than one kernel took rows
    s.Close()
    s2.Close()


@pytest.mark.parametrize("path", [0, 1, 2])
@pytest.mark.parametrize("freq,pres,min_p", [(0.3, 0.4, 0.0), (-0.2, 0.1, 0.0), (0.0, 0.0, 0.05), (0.2, 0.0, 0.02)])
def test_per_row_configurations_with_handle_wide_extras(oracle, rocm, path, freq, pres, min_p):
    # min-p and the frequency / presence penalties stay the handle's while the other settings vary per row
    rng = np.random.default_rng(79)
    B, V, H = 24, 9000, 300
    x = (rng.standard_normal((B, V)) * 2.0).astype(np.float32)
    x[:, :8] += np.float32(3.0)
    u = rng.random(B, dtype=np.float32)
    hist = ((rng.zipf(1.2, size=(B, H)) - 1) % V).astype(np.int32)
    Ts = rng.choice([0.5, 0.7, 1.0, 1.3], B).astype(np.float32)
    ks = rng.choice([0, 1, 5, 40, 64, 65, 128, 129, 300, 512, 700, V], B).astype(np.int32)
    ps = rng.choice([1.0, 0.9, 0.5, 0.99], B).astype(np.float32)
    reps = rng.choice([1.0, 1.15, 2.0, 0.8], B).astype(np.float32)
    s, tok, pr = _sample_rows(rocm, x, u, hist, Ts, ks, ps, reps, path, MinP=min_p, FrequencyPenalty=freq, PresencePenalty=pres)
    s.Status()
    for b in range(B):
        want = oracle.sample(x[b:b + 1], u[b:b + 1], float(Ts[b]), int(ks[b]), float(ps[b]), float(reps[b]), hist[b:b + 1], None,
                             mode=oracle.MODE_FIXED, min_p=min_p, freq=freq, pres=pres)
        assert tok[b] == want["tokens"][0], (b, Ts[b], ks[b], ps[b], reps[b])
        assert pr[b:b + 1].view(np.uint32)[0] == want["probs"].view(np.uint32)[0], b
    if path != 1 and freq < 0:
        # a penalty that raises logits, a history that the single-pass kernel's hash holds: its rows stay its own
        assert s.Counters()["topk_rows"] == int(((ks >= 1) & (ks <= 512)).sum())
    s.Close()


@pytest.mark.parametrize("path", [0, 1, 2])
def test_per_row_min_p_and_additive_penalties(oracle, rocm, path):
    # all seven settings per row; the handle is configured without a frequency / presence penalty, so the call itself
    # brings the table of counts into being
    rng = np.random.default_rng(80)
    B, V, H = 32, 9000, 300
    x = (rng.standard_normal((B, V)) * 2.0).astype(np.float32)
    x[:, :8] += np.float32(3.0)
    u = rng.random(B, dtype=np.float32)
    hist = ((rng.zipf(1.2, size=(B, H)) - 1) % V).astype(np.int32)
    Ts = rng.choice([0.5, 0.7, 1.0, 1.3], B).astype(np.float32)
    ks = rng.choice([0, 1, 5, 40, 64, 65, 128, 129, 300, 512, 700, V], B).astype(np.int32)
    ps = rng.choice([1.0, 0.9, 0.5, 0.99], B).astype(np.float32)
    reps = rng.choice([1.0, 1.15, 2.0, 0.8], B).astype(np.float32)
    mps = rng.choice([0.0, 0.0, 0.01, 0.1, 0.5], B).astype(np.float32)
    frs = rng.choice([0.0, 0.0, 0.2, 1.0, -0.3], B).astype(np.float32)
    prs = rng.choice([0.0, 0.0, 0.4, -0.2], B).astype(np.float32)
    s, tok, pr = _sample_rows(rocm, x, u, hist, Ts, ks, ps, reps, path, min_ps=mps, freqs=frs, press=prs)
    s.Status()
    for b in range(B):
        want = oracle.sample(x[b:b + 1], u[b:b + 1], float(Ts[b]), int(ks[b]), float(ps[b]), float(reps[b]), hist[b:b + 1], None,
                             mode=oracle.MODE_FIXED, min_p=float(mps[b]), freq=float(frs[b]), pres=float(prs[b]))
        assert tok[b] == want["tokens"][0], (b, Ts[b], ks[b], ps[b], reps[b], mps[b], frs[b], prs[b])
        assert pr[b:b + 1].view(np.uint32)[0] == want["probs"].view(np.uint32)[0], b
    s.Close()
    # only the new arrays, everything else from the handle (T 0.9, top_k 7, top_p 0.8, penalty 1.3); a second call on the
    # same handle with other histories finds the table clean
    for rep_call in range(2):
        hist2 = ((rng.zipf(1.2, size=(B, H)) - 1) % V).astype(np.int32)
        s2, tok2, _ = _sample_rows(rocm, x, u, hist2, None, None, None, None, path, min_ps=mps, freqs=frs, press=prs)
        s2.Status()
        s2.Close()
        for b in range(B):
            want = oracle.sample(x[b:b + 1], u[b:b + 1], 0.9, 7, 0.8, 1.3, hist2[b:b + 1], None, mode=oracle.MODE_FIXED,
                                 min_p=float(mps[b]), freq=float(frs[b]), pres=float(prs[b]))
            assert tok2[b] == want["tokens"][0], (rep_call, b)
    # invalid values of the new settings are reported like the others
    bad_mp = mps.copy(); bad_mp[3] = 1.0; bad_mp[5] = -0.1
    bad_fr = frs.copy(); bad_fr[7] = np.inf
    bad_pr = prs.copy(); bad_pr[9] = np.nan
    s3, tok3, _ = _sample_rows(rocm, x, u, hist, Ts, ks, ps, reps, path, min_ps=bad_mp, freqs=bad_fr, press=bad_pr)
    with pytest.raises(rocm.BornRocmError, match="invalid per-row configuration"):
        s3.Status()
    assert tok3[3] == 0 and tok3[5] == 0 and tok3[7] == 0 and tok3[9] == 0
    good = [b for b in range(B) if b not in (3, 5, 7, 9)]
    assert np.array_equal(tok3[good], tok[good])
    s3.Close()


@pytest.mark.parametrize("path", [0, 1, 2])
def test_per_row_promised_kinds_of_row(oracle, rocm, path):
    from born_amd import _capi
    rng = np.random.default_rng(81)
    B, V, H = 20, 9000, 48
    x = (rng.standard_normal((B, V)) * 2.0).astype(np.float32)
    u = rng.random(B, dtype=np.float32)
    hist = rng.integers(0, V, (B, H)).astype(np.int32)
    Ts = rng.choice([0.5, 0.7, 1.0, 1.3], B).astype(np.float32)
    ps = rng.choice([1.0, 0.9, 0.5], B).astype(np.float32)
    reps = rng.choice([1.0, 1.15, 2.0], B).astype(np.float32)

    def want(b, k):
        return oracle.sample(x[b:b + 1], u[b:b + 1], float(Ts[b]), int(k), float(ps[b]), float(reps[b]), hist[b:b + 1], None,
                             mode=oracle.MODE_FIXED)["tokens"][0]

    # every row a small top-k, and the caller says so: only the single-pass kernel runs (under path 1 the general one)
    ks = rng.choice([1, 5, 40, 64, 90, 128, 200, 512], B).astype(np.int32)
    s, tok, _ = _sample_rows(rocm, x, u, hist, Ts, ks, ps, reps, path, row_kinds=_capi.ROWS_SMALL_TOP_K)
    s.Status()
    assert [int(t) for t in tok] == [int(want(b, ks[b])) for b in range(B)]
    c = s.Counters()
    assert (c["general_rows"] == 0) if path != 1 else (c["topk_rows"] + c["fallback_rows"] == 0)
    s.Close()
    # two kinds promised, a third occurs in rows 3 and 11 (top_k 600), and row 7 is invalid: those rows are reported
    ks2 = rng.choice([0, 5, 50], B).astype(np.int32)
    ks2[3] = ks2[11] = 600
    Tbad = Ts.copy()
    Tbad[7] = -1.0
    s, tok, _ = _sample_rows(rocm, x, u, hist, Tbad, ks2, ps, reps, path, row_kinds=_capi.ROWS_SMALL_TOP_K | _capi.ROWS_NO_TOP_K)
    if path != 1:
        with pytest.raises(rocm.BornRocmError, match="invalid per-row configuration"):
            s.Status()
        assert tok[3] == 0 and tok[11] == 0 and tok[7] == 0
        good = [b for b in range(B) if b not in (3, 7, 11)]
    else:                                                # path 1: the general kernel serves every valid row whatever was promised
        with pytest.raises(rocm.BornRocmError, match="invalid per-row configuration"):
            s.Status()
        assert tok[7] == 0
        good = [b for b in range(B) if b != 7]
    assert [int(tok[b]) for b in good] == [int(want(b, ks2[b])) for b in good]
    s.Close()
    with pytest.raises(rocm.SamplerPanic, match="row_kinds"):
        _sample_rows(rocm, x, u, hist, Ts, ks, ps, reps, path, row_kinds=8)


def test_per_row_invalid_configuration_is_reported(oracle, rocm):
    rng = np.random.default_rng(78)
    B, V = 6, 3000
    x = rng.standard_normal((B, V)).astype(np.float32)
    u = rng.random(B, dtype=np.float32)
    Ts = np.array([1.0, 0.0, 1.0, np.nan, 0.7, 1.0], np.float32)
    ps = np.array([0.9, 0.9, 1.5, 0.9, 0.9, 0.0], np.float32)
    ks = np.array([10, 10, 10, 10, 0, 10], np.int32)
    s, tok, pr = _sample_rows(rocm, x, u, None, Ts, ks, ps, None)
    with pytest.raises(rocm.BornRocmError, match="invalid per-row configuration"):
        s.Status()
    for b in (0, 4):                                                         # the valid rows are unaffected
        want = oracle.sample(x[b:b + 1], u[b:b + 1], float(Ts[b]), int(ks[b]), float(ps[b]), 1.3, None, None, mode=oracle.MODE_FIXED)
        assert tok[b] == want["tokens"][0]
    assert tok[[1, 2, 3, 5]].tolist() == [0, 0, 0, 0]
    s.Close()


# ---------------------------------------------------------------- error behaviour

def test_argument_errors_panic_like_the_go_layer(rocm):
    with pytest.raises(rocm.SamplerPanic, match="sampler: temperature"):
        rocm.NewSampler(rocm.SamplerConfig(Temperature=-1.0))
    with pytest.raises(rocm.SamplerPanic, match="top_p"):
        rocm.NewSampler(rocm.SamplerConfig(TopP=-0.5))
    with pytest.raises(rocm.SamplerPanic, match="repetition_penalty"):
        rocm.NewSampler(rocm.SamplerConfig(RepetitionPenalty=float("nan")))
    with pytest.raises(rocm.SamplerPanic):
        rocm.NewSampler(max_batch=0)
    s = rocm.NewSampler(max_batch=4, max_vocab=100)
    cfg = s.Config()
    assert (cfg.Temperature, cfg.TopK, cfg.TopP, cfg.RepetitionPenalty) == (1.0, 0, 1.0, 1.0)      # zero => defaults
    buf = rocm.DeviceBuffer(4 * 4 * 100)
    tok = rocm.DeviceBuffer(16)
    with pytest.raises(rocm.SamplerPanic, match="exceeds"):
        s.Sample(buf, 5, 100, None, None, None, tok)
    with pytest.raises(rocm.SamplerPanic, match="row_stride"):
        s.Sample(buf, 4, 100, None, None, None, tok, row_stride=50)
    with pytest.raises(rocm.SamplerPanic, match="null"):
        s.Sample(None, 4, 100, None, None, None, tok)
    with pytest.raises(rocm.SamplerPanic, match="> 0"):
        s.Sample(buf, 0, 100, None, None, None, tok)
    # out-of-range history ids: ignored by the kernel, reported by Status
    x = np.random.default_rng(0).standard_normal((4, 100), dtype=np.float32)
    h = np.array([[1, 2, 300, -4]] * 4, np.int32)
    s.SetConfig(rocm.SamplerConfig(TopK=10, RepetitionPenalty=1.2))
    rocm.sample_host(s, x, np.full(4, 0.5, np.float32), h)
    with pytest.raises(rocm.BornRocmError, match="history"):
        s.Status()


# ---------------------------------------------------------------- the benchmark configurations

def test_config_c1_steps(oracle, rocm):
    """C1: batch 1, vocab 32000, fresh logits per step; 200 of the 1000 steps (every fifth) against both oracle layers."""
    from born_amd import synth
    s = rocm.NewSampler(rocm.SamplerConfig(Temperature=0.8, TopK=40, TopP=0.95, RepetitionPenalty=1.1), max_batch=1,
                        max_vocab=32000)
    near = 0
    for step in range(0, 1000, 5):
        w = synth.c1(step)
        got = rocm.sample_host(s, w.logits, w.uniforms, w.history)
        fx = oracle.sample(w.logits, w.uniforms, 0.8, 40, 0.95, 1.1, w.history, mode=oracle.MODE_FIXED)
        tr = oracle.sample(w.logits, w.uniforms, 0.8, 40, 0.95, 1.1, w.history, mode=oracle.MODE_TRUTH)
        assert got["tokens"][0] == fx["tokens"][0] and got["probs"][0] == fx["probs"][0], step
        assert got["tokens"][0] == tr["tokens"][0] or tr["near"][0]
        near += int(tr["near"][0])
    assert near <= 6


def test_config_c2_greedy_and_multinomial(oracle, rocm):
    from born_amd import synth
    w = synth.c2()
    assert np.array_equal(_argmax(rocm, w.logits), oracle.argmax_ref(w.logits))
    got, _, tr = _check_against_oracle(oracle, rocm, w.logits, w.uniforms)          # T=1, full vocabulary
    assert got["counters"]["general_rows"] == 64
    assert tr["near"].sum() <= 4


@pytest.mark.parametrize("path", TOPK_PATHS)
def test_config_c3_full_batch(oracle, rocm, path):
    """The benchmark configuration at full size: all 256 rows bit-exact against the fixed-point layer,
    equal to the fp64 truth except on flagged rows, every row served by the single-pass path."""
    from born_amd import synth
    w = synth.c3()
    got, _, tr = _check_against_oracle(oracle, rocm, w.logits, w.uniforms, w.temperature, w.top_k, w.top_p, w.rep,
                                       w.history, nuc=64, path=path)
    c = got["counters"]
    assert c["topk_rows"] == 256 and c["fallback_rows"] == 0 and c["general_rows"] == 0
    print(f"C3: rows flagged near a CDF step by the truth layer: {int(tr['near'].sum())} of 256, "
          f"tokens differing from the truth layer: {int((got['tokens'] != tr['tokens']).sum())}")
    assert tr["near"].sum() <= 3


def test_config_c4_full(oracle, rocm):
    from born_amd import synth
    w = synth.c4()
    e = w.extra
    s = rocm.NewSampler(max_batch=64, max_vocab=32000)
    got = rocm.verify_host(s, e["target"], e["draft"], e["draft_tokens"], e["u_acc"], e["u_res"])
    fx = oracle.spec_verify(e["target"], e["draft"], e["draft_tokens"], e["u_acc"], e["u_res"], mode=oracle.MODE_FIXED)
    tr = oracle.spec_verify(e["target"], e["draft"], e["draft_tokens"], e["u_acc"], e["u_res"], mode=oracle.MODE_TRUTH)
    assert np.array_equal(got["n_accepted"], fx["n_accepted"]) and np.array_equal(got["next_token"], fx["next_token"])
    diff = (got["n_accepted"] != tr["n_accepted"]) | (got["next_token"] != tr["next_token"])
    assert not (diff & ~tr["near"]).any()
    # residual CDF steps are ~3e-5 wide at this vocabulary, so a few of the 64 draws land within 1e-6 of one
    assert tr["near"].sum() <= 8
    print(f"C4: {int(tr['near'].sum())} of 64 sequences flagged near a boundary, {int(diff.sum())} differ from the truth layer")
    # every sequence either accepted everything or carries a resampled token of the vocabulary
    full = got["n_accepted"] == 5
    assert np.all(got["next_token"][full] == -1) and np.all((got["next_token"][~full] >= 0) & (got["next_token"][~full] < 32000))


def test_config_c5_slice_and_full_size_properties(oracle, rocm):
    """C5 (wide nucleus, vocabulary 152064): 64 rows from across the batch against the oracle; the full 1024-row batch
    through size-independent properties (determinism, row independence, range)."""
    from born_amd import synth
    w = synth.c5(rows=1024)
    B, V = w.logits.shape
    s = rocm.NewSampler(rocm.SamplerConfig(Temperature=w.temperature, TopP=w.top_p, RepetitionPenalty=w.rep),
                        max_batch=B, max_vocab=V)
    full = rocm.sample_host(s, w.logits, w.uniforms, w.history)
    again = rocm.sample_host(s, w.logits, w.uniforms, w.history)
    assert np.array_equal(full["tokens"], again["tokens"]) and np.array_equal(full["probs"], again["probs"])
    assert full["tokens"].min() >= 0 and full["tokens"].max() < V and np.all(full["probs"] > 0)
    sl = slice(500, 524)
    part = rocm.sample_host(s, w.logits[sl], w.uniforms[sl], w.history[sl])
    assert np.array_equal(part["tokens"], full["tokens"][sl])                       # rows are independent
    assert np.array_equal(part["probs"].view(np.uint32), full["probs"][sl].view(np.uint32))
    # 64 rows drawn across the batch (its first and last eight and 48 others) against both oracle layers
    rng = np.random.default_rng(synth.BASE_SEED + 5)
    idx = np.unique(np.concatenate([np.arange(8), np.arange(B - 8, B), rng.choice(np.arange(8, B - 8), 48, replace=False)]))
    x, u, h = np.ascontiguousarray(w.logits[idx]), w.uniforms[idx], np.ascontiguousarray(w.history[idx])
    fx = oracle.sample(x, u, w.temperature, 0, w.top_p, w.rep, h, mode=oracle.MODE_FIXED)
    tr = oracle.sample(x, u, w.temperature, 0, w.top_p, w.rep, h, mode=oracle.MODE_TRUTH)
    got_t, got_p = full["tokens"][idx], full["probs"][idx]
    assert np.array_equal(got_t, fx["tokens"])
    assert np.array_equal(got_p.view(np.uint32), fx["probs"].view(np.uint32))
    diff = got_t != tr["tokens"]
    assert not (diff & ~tr["near"]).any()
    # CDF steps are about 1e-5 wide on these flat rows, so the 1e-6 criterion flags many rows by itself; what is held
    # to a bound is the number of tokens that actually differ from the fp64 layer (a draw within ~3e-7 of a step)
    assert int(diff.sum()) <= 4, f"{int(diff.sum())} of {idx.size} tokens differ from the fp64 layer"
    assert np.allclose(got_p[~diff], tr["probs"][~diff], rtol=1e-5)
    print(f"C5: {int(tr['near'].sum())} of {idx.size} rows flagged near a CDF step, {int(diff.sum())} tokens differ from the truth layer")
    s.Status()
