// Sampler for top_k disabled (full-vocabulary multinomial and top-p): one workgroup of 1024 or 512 threads per
// row, three sweeps over the row (docs/SAMPLING_SPEC.md, fixed-point layer).
//
//   sweep 1  maximum and smallest finite value of the penalised logits (z is a non-decreasing function of
//            the penalised logit, so no division is needed yet): m = z(max), and the span of d = m - z.
//   sweep 2  integer masses trunc(expneg(d) * 2^S) accumulated into 4096 bins that cover exactly that span
//            (u64 LDS atomics), then an inclusive scan: cumulative mass in rank order, bin by bin.
//   targets  the top-p cut target ceil(p * Z) falls into one bin, the draw's into one of the few that the interval of
//            the nucleus's mass allows: one gather serves both.
//   sweep 3  gather: a compare of the penalised logit against the wanted bins' value ranges (widened, so
//            that it can only over-select) stages about 1 % of the row in per-wave LDS lists (ballot + lane
//            rank); the staged entries are then classified exactly.
//   resolve  the gathered entries are put in rank order through buckets, one scan of their masses gives every entry
//            the mass at and above it within its bin (a short list: summed directly); the first entry in rank
//            order whose cumulative mass reaches a target is the one whose own mass crosses it.
// A wanted bin too full for the lists (heavy ties) is refined in place by a radix descent over
// the rank keys of that bin, 11 bits per sweep.
// In the usual row (a maximum of ordinary size, a temperature whose division has the three-instruction shortcut, no
// min-p bound, a history short enough to be listed) sweeps 2 and 3 read the logits as stored: no history bitmap, no
// test of a logit's magnitude, clamps in place of selects; what the seen ids contribute is corrected apart (the
// histogram is a sum of integers, so a stored logit's mass comes out again exactly).  The sweeps are then bound by
// the three reads of the row from HBM, not by the vector ALU.
#pragma once
#include <algorithm>
#include <type_traits>
#include "dev_common.h"
#include "finish.h"
#include "kernels.h"
#include "row_config.h"

namespace born {

// Threads per row: 1024 (one workgroup per CU: the shortest time per row, for batches that leave CUs idle anyway) or
// 512 (two workgroups per CU: one row's sweeps that wait for memory overlap the other's sweep that computes; for
// batches of more rows than the device has CUs). The geometry below follows from it.
constexpr int NUC_BINS = 4096;
constexpr int NUC_BEYOND = 16;                // slots behind the bins, for what lies beyond the last one
constexpr int NUC_DIRECT = 32;                // listed entries that sum what ranks above them directly
template <int BLOCK>
struct NucGeom {
    static_assert(BLOCK == 512 || BLOCK == 1024, "threads per row");
    static constexpr int WAVES = BLOCK / WAVE;
    static constexpr int U = 4;                                   // 128-bit loads per thread and stage (more in flight measured slower)
    static constexpr int WCAP = BLOCK == 1024 ? 160 : 256;       // staged entries per wave
    static constexpr int CAP = BLOCK;                             // gathered entries (one per thread)
    static constexpr int PER = NUC_BINS / BLOCK;                  // bins per thread in the scan
    static constexpr int SUB = 2048 / BLOCK;                      // sub-bins per thread in a radix-descent scan
    static_assert(WAVES * WCAP >= 2048 && CAP * 4 >= 2048, "the sub-histograms fit the list storage");
};

typedef row_f32x4 nuc_f32x4;

struct NucRow {                               // uniform per workgroup
    const float *x;
    int V, n4;                                // n4: the blocks of four that are read by 128-bit loads
    bool penal, degenerate;
    bool masked = false;                      // the visitor replaces every seen logit by `skip`; the seen ids are visited apart
    float skip = 0.0f;
    float T, rcp, rep, m, scale, range, sbin, dcut;        // rcp: RN(1 / T) where the division shortcut is exact, else 0
    const unsigned *counts;                   // occurrences of each id in the row's history (frequency / presence penalties), or null
    float freq, pres;
};

__device__ __forceinline__ float nuc_z(const NucRow &r, float y) {
    if (r.T == 1.0f) return canon(y);
    return canon(y / r.T);
}
__device__ __forceinline__ float nuc_d(const NucRow &r, float z) { return r.degenerate ? 0.0f : r.m - z; }
__device__ __forceinline__ int nuc_bin(const NucRow &r, float d) {
    return (int)fminf(d * r.sbin, (float)(NUC_BINS - 1));          // monotone in d; NaN, inf and all beyond the span -> last bin
}
// (the magnitude test of the division shortcut and of the unit-temperature path: dev_common.h)
__device__ __forceinline__ bool nuc_ordinary(float y) { return ordinary_magnitude(y); }
// ANY_T: a row's own temperature, which the host has not seen.  The first correction's quotient lies within a hair of half
// an ulp of y / T whatever T is (the start is off by an ulp and a half at most, the correction leaves 2^-23 of that), so
// the second residual is exact and, with rcp = RN(1 / T), the second correction gives the correctly rounded quotient for every T
// (Markstein's theorem: a quotient within an ulp, corrected once with a correctly rounded reciprocal).  Five instructions
// where the division takes eleven and keeps the row from the arithmetic of usual rows.
template <bool ANY_T>
__device__ __forceinline__ float nuc_z_shortcut(const NucRow &r, float y) {
    float q = __fmul_rn(y, r.rcp);
    if (ANY_T) q = __fmaf_rn(__fmaf_rn(-q, r.T, y), r.rcp, q);
    const float e = __fmaf_rn(-q, r.T, y);
    return __fmaf_rn(e, r.rcp, q);
}
// RN(1 / T) for ANY_T; 0 where the division is taken: T = 1 needs none, outside [2^-20, 2^20] a residual may underflow.
__device__ __forceinline__ float nuc_reciprocal(float T) {
    return T >= 0x1p-20f && T <= 0x1p20f && T != 1.0f ? uniform_f32(1.0f / T) : 0.0f;
}

// Visits every element of the row with its penalised logit: four at a time as f4(id of the first, y[4]), in stages of
// U float4 per thread, the next stage's loads in flight while this one is visited; what is left over (and every element of a
// short row that is not aligned) one at a time as f1(id, y).
// AHEAD: the row's partial last stage is loaded ahead like the whole ones (3 % faster on short rows, where the few
// blocks left over are a third of the row; measured slower on long ones and in the single-sweep kernel).
// `pre` runs once before the first element is visited, with the first stage's loads already in flight (work that
// must precede the visits but not the loads: building the history bitmap).
struct NucNoPre {
    __device__ __forceinline__ void operator()() const {}
};
// NT: the row is read once (non-temporal loads: measured 6 % faster for a single sweep); a kernel that sweeps the row
// again wants it to stay in the caches.
// The block of four logits `off` bytes behind block b of the row.  x and b are uniform: the row's address and the stage's are added in scalar registers,
// and a lane holds one 32-bit offset for all its loads (512 threads: 88 registers, 128 with an offset per load).
static_assert(WIDE_MAX_VOCAB < (1 << 30), "a row's bytes fit 32 bits");
template <bool NT>
__device__ __forceinline__ nuc_f32x4 nuc_load4(const float *x, int b, u32 off) {
    const nuc_f32x4 *p = reinterpret_cast<const nuc_f32x4 *>(reinterpret_cast<const char *>(x) + (u32)b * 16u + off);
    return NT ? __builtin_nontemporal_load(p) : *p;
}
// This thread's block of the workgroup's blocks from b on, or the row's last block beyond it.
template <bool NT>
__device__ __forceinline__ nuc_f32x4 nuc_load4_clamped(const float *x, int b, int last) {
    const int from = min(b, last);
    return nuc_load4<NT>(x, from, min((u32)threadIdx.x, (u32)(last - from)) * 16u);
}
// PLAIN: the caller knows that the row has no penalties (a loop of its own without the penalty code: the visitor's
// test of r.penal at every visit cost the single-sweep kernel 5 %).
// LOADS_FIRST: a stage's loads are issued before the visits of the one before, not among them, where the compiler spilled registers for them; off for
// the sweep of token_logprob_kernel, whose single rows it holds up (1 x 50 257: 10.2 us, 9.9 without; 1024 x 152 064 101.5 and 101.9).
// FIRST (AHEAD instances only): `first` holds the row's first stage, requested earlier with nuc_request_first, or
// (NucKept) its first blocks, kept in registers from the first sweep on, which fills them (NucFill).
struct NucNoFirst {};
template <int NUC_BLOCK>
struct NucKept {
    static constexpr int LOADS = NUC_BLOCK == 512 ? 10 : NucGeom<NUC_BLOCK>::U;   // of a thread: what the 128 registers of a lane leave (1024: a stage)
    nuc_f32x4 v[LOADS];
};
template <int NUC_BLOCK>
struct NucFill {
    NucKept<NUC_BLOCK> *kept;
};
template <int NUC_BLOCK, bool NT = false, bool AHEAD = false, bool PLAIN = false, bool LOADS_FIRST = true, class F4, class F1, class PRE = NucNoPre,
          class FIRST = NucNoFirst>
__device__ __forceinline__ void nuc_foreach4(const NucRow &r, const u32 *bm, F4 f4, F1 f1, PRE pre = PRE(),
                                             const FIRST &first = FIRST()) {
    const int tid = threadIdx.x;
    auto visit4 = [&](const nuc_f32x4 &q, int j) {
        float y[4] = {q[0], q[1], q[2], q[3]};
        if (!PLAIN && r.penal) {
            // One seen element per turn, the lowest first: with a long history nearly every wave has some lane with a seen
            // id among its four, but a lane rarely holds two, so the wave computes one penalty per visit, not four.
            u32 bits = (bm[j >> 5] >> (j & 31)) & 0xFu;
            if (r.masked) {
                // a sign-extended bit field extract and a bitwise select per element, unconditionally: a branch around
                // them is taken by nearly every wave once the history has a few hundred ids
                const u32 sk = __float_as_uint(r.skip);
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    const u32 m = (u32)((int)(bits << (31 - t)) >> 31);
                    y[t] = __uint_as_float((sk & m) | (__float_as_uint(y[t]) & ~m));
                }
                bits = 0u;
            }
            while (bits) {
                const u32 low = bits & (0u - bits);
                const float v = low == 1u ? y[0] : low == 2u ? y[1] : low == 4u ? y[2] : y[3];
                const float pv = penalise_seen(v, r.rep, r.counts, j + (31 - __clz(low)), r.freq, r.pres);
                y[0] = low == 1u ? pv : y[0];
                y[1] = low == 2u ? pv : y[1];
                y[2] = low == 4u ? pv : y[2];
                y[3] = low == 8u ? pv : y[3];
                bits ^= low;
            }
        }
        f4(j, y);
    };
    auto visit1 = [&](int j) {
        float y = r.x[j];
        if (!PLAIN && r.penal && ((bm[j >> 5] >> (j & 31)) & 1u)) y = r.masked ? r.skip : penalise_seen(y, r.rep, r.counts, j, r.freq, r.pres);
        f1(j, y);
    };
    const int n4 = r.n4;
    constexpr int NUC_U = NucGeom<NUC_BLOCK>::U, NUC_KEPT = NucKept<NUC_BLOCK>::LOADS;
    constexpr bool FILL = std::is_same<FIRST, NucFill<NUC_BLOCK>>::value, KEPT = FILL || std::is_same<FIRST, NucKept<NUC_BLOCK>>::value;
    if constexpr (!AHEAD) {
        const int kept_blocks = KEPT && n4 >= (NUC_KEPT + NUC_U) * NUC_BLOCK ? NUC_KEPT * NUC_BLOCK : 0;
        const int nfull = (n4 - kept_blocks) / (NUC_U * NUC_BLOCK);
        if (nfull > 0) {
            // Two stages a turn, each loaded while the other is visited, so that no register is copied; the last
            // one or two stages in a loop of their own.
            nuc_f32x4 va[NUC_U], vb[NUC_U];
            const u32 off = (u32)tid * 16u;
            int s = 0;
            if constexpr (FILL) {
                if (kept_blocks)
#pragma unroll
                    for (int k = 0; k < NUC_KEPT; k++) first.kept->v[k] = nuc_load4<NT>(r.x, k * NUC_BLOCK, off);
            }
#pragma unroll
            for (int u = 0; u < NUC_U; u++) va[u] = nuc_load4<NT>(r.x, kept_blocks + (s * NUC_U + u) * NUC_BLOCK, off);
            pre();
            if constexpr (KEPT) {
                const NucKept<NUC_BLOCK> *kept;
                if constexpr (FILL) kept = first.kept;
                else kept = &first;
                if (kept_blocks)
#pragma unroll
                    for (int k = 0; k < NUC_KEPT; k++) visit4(kept->v[k], (k * NUC_BLOCK + tid) << 2);
            }
            for (; s + 2 < nfull; s += 2) {
#pragma unroll
                for (int u = 0; u < NUC_U; u++) vb[u] = nuc_load4<NT>(r.x, kept_blocks + ((s + 1) * NUC_U + u) * NUC_BLOCK, off);
                if (LOADS_FIRST) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int u = 0; u < NUC_U; u++) visit4(va[u], (kept_blocks + (s * NUC_U + u) * NUC_BLOCK + tid) << 2);
#pragma unroll
                for (int u = 0; u < NUC_U; u++) va[u] = nuc_load4<NT>(r.x, kept_blocks + ((s + 2) * NUC_U + u) * NUC_BLOCK, off);
                if (LOADS_FIRST) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int u = 0; u < NUC_U; u++) visit4(vb[u], (kept_blocks + ((s + 1) * NUC_U + u) * NUC_BLOCK + tid) << 2);
            }
            for (;;) {
#pragma unroll
                for (int u = 0; u < NUC_U; u++) visit4(va[u], (kept_blocks + (s * NUC_U + u) * NUC_BLOCK + tid) << 2);
                if (++s >= nfull) break;
#pragma unroll
                for (int u = 0; u < NUC_U; u++) va[u] = nuc_load4<NT>(r.x, kept_blocks + (s * NUC_U + u) * NUC_BLOCK, off);
            }
        } else {
            pre();
        }
        for (int i = kept_blocks + nfull * NUC_U * NUC_BLOCK + tid; i < n4; i += NUC_BLOCK) {
            const nuc_f32x4 q = nuc_load4<NT>(r.x, 0, (u32)i * 16u);
            visit4(q, i << 2);
        }
    } else {
        const int nst = (n4 + NUC_U * NUC_BLOCK - 1) / (NUC_U * NUC_BLOCK);      // stages, the last one whole or partial
        if (nst > 0) {
            // Loads are unconditional, of a block index clamped to the row's last block (a load under a condition makes
            // the compiler wait for every load in flight); only the visits of the last stage ask whether the block exists.
            nuc_f32x4 va[NUC_U], vb[NUC_U];
            const int lastb = n4 - 1;
            int s = 0;
            if constexpr (FILL) {
#pragma unroll
                for (int u = 0; u < NUC_U; u++) first.kept->v[u] = nuc_load4_clamped<NT>(r.x, u * NUC_BLOCK, lastb);
            }
            if constexpr (!KEPT && !std::is_same<FIRST, NucNoFirst>::value) {
#pragma unroll
                for (int u = 0; u < NUC_U; u++) va[u] = first[u];
            } else {
#pragma unroll
                for (int u = 0; u < NUC_U; u++) va[u] = nuc_load4_clamped<NT>(r.x, ((KEPT ? 1 : 0) * NUC_U + u) * NUC_BLOCK, lastb);
            }
            pre();
            if constexpr (KEPT) {
                const NucKept<NUC_BLOCK> *kept;
                if constexpr (FILL) kept = first.kept;
                else kept = &first;
#pragma unroll
                for (int u = 0; u < NUC_U; u++)
                    if (u * NUC_BLOCK + tid < n4) visit4(kept->v[u], (u * NUC_BLOCK + tid) << 2);
                s = 1;
            }
            for (; s + 1 < nst; s++) {
#pragma unroll
                for (int u = 0; u < NUC_U; u++) vb[u] = nuc_load4_clamped<NT>(r.x, ((s + 1) * NUC_U + u) * NUC_BLOCK, lastb);
                if (LOADS_FIRST) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int u = 0; u < NUC_U; u++) visit4(va[u], ((s * NUC_U + u) * NUC_BLOCK + tid) << 2);
#pragma unroll
                for (int u = 0; u < NUC_U; u++) va[u] = vb[u];
            }
            if (!KEPT || nst > 1) {
#pragma unroll
                for (int u = 0; u < NUC_U; u++) {
                    const int i = ((nst - 1) * NUC_U + u) * NUC_BLOCK + tid;
                    if (i < n4) visit4(va[u], i << 2);
                }
            }
        } else {
            pre();
        }
    }
    for (int j = (n4 << 2) + tid; j < r.V; j += NUC_BLOCK) visit1(j);
}
// Requests the first stage of the row's next sweep (the same loads the AHEAD visitor starts with): issued at the
// end of one sweep, they are in flight through the reductions and scans between the sweeps, which on a batch that leaves
// CUs idle are otherwise a memory latency each.
template <int NUC_BLOCK, bool NT>
__device__ __forceinline__ void nuc_request_first(const NucRow &r, nuc_f32x4 (&first)[NucGeom<NUC_BLOCK>::U]) {
    const int n4 = r.n4;
    if (n4 > 0) {
#pragma unroll
        for (int u = 0; u < NucGeom<NUC_BLOCK>::U; u++) first[u] = nuc_load4_clamped<NT>(r.x, u * NUC_BLOCK, n4 - 1);
    }
}
// Visits every element of the row as f(id, penalised logit).
template <int NUC_BLOCK, bool NT = false, bool AHEAD = false, bool PLAIN = false, class F, class PRE = NucNoPre, class FIRST = NucNoFirst>
__device__ __forceinline__ void nuc_foreach(const NucRow &r, const u32 *bm, F f, PRE pre = PRE(), const FIRST &first = FIRST()) {
    nuc_foreach4<NUC_BLOCK, NT, AHEAD, PLAIN>(r, bm, [&](int j, const float (&y)[4]) {
#pragma unroll
        for (int t = 0; t < 4; t++) f(j + t, y[t]);
    }, f, pre, first);
}

// A wave's list of the logits that a sweep wants, (bits, id) each, at most `cap`; what would go beyond is only counted.  The count lives in LDS, not in a register
// of every lane: the row visitor lets lanes of a wave sit out visits (the row's last whole blocks of four end inside a wave, its
// ragged tail starts again at lane 0), and a lane that missed an append must not reuse a position.  LDS operations of one wave complete in order.
// (Relaxed atomic accesses: re-read at every visit as a volatile would be, but they keep the LDS address space, where a volatile access became a flat one
// that waits for the row's loads in flight.)
// The lanes whose y is in [lo, hi] or a NaN, as a mask in scalar registers.
__device__ __forceinline__ u64 nuc_within(float y, float lo, float hi) {
    constexpr int UGE = 11, ULE = 13;                                // (the compare's predicates: true for a NaN)
    return __builtin_amdgcn_fcmpf(y, lo, UGE) & __builtin_amdgcn_fcmpf(y, hi, ULE);
}
struct NucList {
    uint2 *at;
    u32 *count;
    __device__ __forceinline__ void clear() const {
        if (lane_id() == 0) __hip_atomic_store(count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    }
    __device__ __forceinline__ u32 size() const { return __hip_atomic_load(count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT); }
    // mk: the lanes whose logit is wanted
    template <int CAP>
    __device__ __forceinline__ void append(u64 mk, float y, int j) const {
        if (mk) {                                                    // uniform over the lanes that take part in this visit
            const u32 base = size();
            put<CAP>(mk, base, y, j);
            __hip_atomic_store(count, base + (u32)__popcll(mk), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);   // (every lane the same)
        }
    }
    // Four logits of a lane: one branch for the wave's 256, one read of the count.  (A test and a branch per logit were 5 vector instructions
    // and a wait for the compare.)
    template <int CAP, class P>
    __device__ __forceinline__ void append4(P wanted, const float (&y)[4], int j) const {
        const u64 mk[4] = {wanted(y[0]), wanted(y[1]), wanted(y[2]), wanted(y[3])};
        if (mk[0] | mk[1] | mk[2] | mk[3]) {
            u32 base = size();
#pragma unroll
            for (int t = 0; t < 4; t++) {
                if (mk[t]) {
                    put<CAP>(mk[t], base, y[t], j + t);
                    base += (u32)__popcll(mk[t]);
                }
            }
            __hip_atomic_store(count, base, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        }
    }
    template <int CAP>
    __device__ __forceinline__ void put(u64 mk, u32 base, float y, int j) const {
        const u32 pos = base + __builtin_amdgcn_mbcnt_hi((u32)(mk >> 32), __builtin_amdgcn_mbcnt_lo((u32)mk, 0u));
        if (__builtin_amdgcn_inverse_ballot_w64(mk) && pos < (u32)CAP) at[pos] = make_uint2(__float_as_uint(y), (u32)j);
    }
};

// smallest bin whose inclusive cumulative mass reaches target (the last bin if none does); called by whole waves.
// Two rounds of 64 lanes: which run of 64 bins, then which bin of the run (a binary search is twelve dependent LDS reads).
static_assert(NUC_BINS == WAVE * WAVE, "two rounds of one wave cover the bins");
__device__ __forceinline__ int nuc_first_reaching(const u64 *cum, u64 target) {
    const int l = lane_id();
    const u64 runs = __ballot(cum[l * WAVE + WAVE - 1] >= target);
    const int c = runs ? __builtin_ctzll(runs) : WAVE - 1;
    const u64 bins = __ballot(cum[c * WAVE + l] >= target);
    return c * WAVE + (bins ? __builtin_ctzll(bins) : WAVE - 1);
}

// Range of penalised logits that can fall into bin w, widened so that it can only over-select.
__device__ __forceinline__ void nuc_range(const NucRow &r, int w, float &ylo, float &yhi) {
    if (r.degenerate) {
        ylo = -INFINITY;
        yhi = INFINITY;
        return;
    }
    const float dlo = (float)w / r.sbin, dhi = (float)(w + 1) / r.sbin;
    // With u = 2^-24: a logit of the bin has m - z within 3 u of [dlo, dhi] (the difference, its product with sbin, the quotient here), the bounds of z are off by
    // 2 u (|m| + dhi), those of y by 2 u |y| and, where z or y is subnormal, by less than 1e-30.  Not wider than that asks for: in a row whose bins are narrow, of logits that
    // hardly differ, what is staged beside a bin overflows the lists (with 1e-4 of z, 128 x 152 064 of a spread of 0.01: 203 us, 52 so).
    const float sl = 1e-6f * (fabsf(r.m) + dhi);
    const float zhi = r.m - dlo + sl, zlo = r.m - dhi - sl;
    yhi = zhi * r.T;
    ylo = zlo * r.T;
    yhi += 1e-6f * fabsf(yhi) + 1e-30f;
    ylo -= 1e-6f * fabsf(ylo) + 1e-30f;
    if (w == NUC_BINS - 1) ylo = -INFINITY;                          // the last bin also takes everything beyond the span
    if (w == 0) yhi = INFINITY;
}

// cfg_T, cfg_p, cfg_rep: the row's temperature, top_p and repetition penalty (the handle's, or the row's own).
// COUNTED: a frequency or presence penalty is on (the table of occurrence counts is read for ids the history holds);
// its own instance, so that the usual one carries none of it.
// ANY_T: cfg_rcp is the reciprocal of a temperature that the host has not tried the three-instruction quotient on.
// KEEP: the row's first logits (80 KiB of them with 512 threads, 64 with 1024) stay in registers from sweep 1 on.  The sweeps are bound by the row's three reads, of which
// two are that much shorter, and begin without a wait.  (Before, sweeps 2 and 3 had their first stage requested ahead with 1024 threads.  us, then and now:
// 256 x 128 256 63.4 and 61.7; with 512 threads 1024 x 152 064 299.8 and 276.4, 281.1 with 64 KiB, 512 x 50 257 51.3 and 43.5.)
template <int NUC_BLOCK, bool COUNTED, bool KEEP = true, bool ANY_T = false>
__device__ __forceinline__ void nucleus_row_body(const SampleArgs &a, const float cfg_T, const float cfg_p, const float cfg_rep,
                                                 const float cfg_dcut, const float cfg_freq, const float cfg_pres,
                                                 const float cfg_rcp) {
    constexpr int NUC_WAVES = NucGeom<NUC_BLOCK>::WAVES, NUC_WCAP = NucGeom<NUC_BLOCK>::WCAP, NUC_CAP = NucGeom<NUC_BLOCK>::CAP,
                  NUC_PER = NucGeom<NUC_BLOCK>::PER, NUC_SUB = NucGeom<NUC_BLOCK>::SUB;
    extern __shared__ __align__(16) u64 nuc_dyn[];
    __shared__ BlockScratch scr;
    __shared__ int s_n, s_over, s_nseen;
    __shared__ u64 s_win[2], s_mass[2], s_slot0[2];
    __shared__ u32 s_wcount[NUC_WAVES], s_top[2], s_low[2];

    u64 *const mass = nuc_dyn;                                                   // [NUC_BINS] masses, then cumulative; [NUC_BEYOND] more until the scan, in the lists
    uint2 *const stage = reinterpret_cast<uint2 *>(nuc_dyn + NUC_BINS);          // [NUC_WAVES][NUC_WCAP] (logit bits, id)
    u64 *const fkey = nuc_dyn + NUC_BINS + NUC_WAVES * NUC_WCAP;                 // [NUC_CAP] rank keys of the gathered entries
    u64 *const fq = fkey + NUC_CAP;                                              // [NUC_CAP] mass | slot << 62
    u32 *const bm = reinterpret_cast<u32 *>(fq + NUC_CAP);                       // history bitmap, one bit per id

    const int tid = threadIdx.x, row = blockIdx.x;
    const int V = a.V;

    NucRow r;
    r.x = a.logits + (long long)row * a.row_stride;
    r.V = V;
    r.n4 = a.row_blocks;
    r.T = cfg_T;
    r.rcp = cfg_rcp;
    r.rep = cfg_rep;
    r.scale = mass_scale(a.mass_shift);
    r.dcut = cfg_dcut;
    const float u = a.uniforms ? a.uniforms[row] : uniform_of(a.seed, a.step, (u64)row);

    BORN_STAMP(a, row, 0);
    // ---- history bitmap
    const int hlen = a.history ? min((int)(a.hist_len ? a.hist_len[row] : (int)a.hist_stride), (int)a.hist_stride) : 0;
    const int *h = a.history + (long long)row * a.hist_stride;
    r.counts = COUNTED ? a.hist_counts + (long long)row * V : nullptr;
    r.freq = COUNTED ? cfg_freq : 0.0f;
    r.pres = COUNTED ? cfg_pres : 0.0f;
    r.penal = (cfg_rep != 1.0f || COUNTED) && hlen > 0;
    constexpr int NUC_SEEN = 4;
    u32 *const seen_list = reinterpret_cast<u32 *>(fkey);            // [NUC_SEEN * NUC_BLOCK], free until the gather classifies
    static_assert(NUC_SEEN * NUC_BLOCK * sizeof(u32) <= 2 * NUC_CAP * sizeof(u64), "the list of seen ids fits the gathered entries' storage");
    const bool list_seen = r.penal && hlen <= NUC_SEEN * NUC_BLOCK;
    int seen_id[NUC_SEEN];
    float seen_y[NUC_SEEN], seen_raw[NUC_SEEN];
    bool lin = false;
    r.masked = list_seen;
    r.skip = -INFINITY;                                              // sweep 1: neither the maximum nor the smallest finite value
    // What must precede the first visit of sweep 1 but not its first loads: run by the row visitor with the first stage
    // in flight (barriers that wait for LDS only).
    auto prologue = [&]() {
        if (r.penal)
            for (int i = tid; i < ((V + 31) >> 5); i += NUC_BLOCK) bm[i] = 0u;
        for (int i = tid; i < NUC_BINS; i += NUC_BLOCK) mass[i] = 0ull;
        if (tid < NUC_BEYOND) mass[NUC_BINS + tid] = 0ull;
        if (tid == 0) {
            s_n = 0;
            s_over = 0;
            s_win[0] = s_win[1] = 0ull;
            s_nseen = 0;
        }
        lds_barrier();
        // The ids the history holds, each once (whoever sets an id's bit first lists it): at most NUC_SEEN per thread, kept
        // in registers with their penalised logits for the whole kernel. The sweeps then see a constant in place of a seen
        // logit (chosen per sweep so that it contributes nothing) and visit the seen ids apart, every lane busy; applying the
        // penalty inside the sweep costs a whole wave the penalty arithmetic whenever one of its lanes holds a seen id, which
        // with a long history is nearly always. A history too long for the registers keeps the penalty inside the sweeps.
        if (list_seen) {
            int hv[NUC_SEEN];                                            // (all of the thread's history loads in flight together)
#pragma unroll
            for (int k = 0; k < NUC_SEEN; k++) {
                const int i = tid + k * NUC_BLOCK;
                hv[k] = i < hlen ? h[i] : -2;
            }
#pragma unroll
            for (int k = 0; k < NUC_SEEN; k++) {
                const int t = hv[k];
                bool first = false;
                if (t >= 0 && t < V) {
                    const u32 bit = 1u << (t & 31);
                    const u32 old = atomicOr(&bm[t >> 5], bit);
                    first = !(old & bit);
                } else if (t != -2) {
                    atomicOr(a.status, 1);
                }
                // one addition to the list's length per wave
                const u64 mk = __ballot(first);
                if (mk) {
                    const u32 rank = __builtin_amdgcn_mbcnt_hi((u32)(mk >> 32), __builtin_amdgcn_mbcnt_lo((u32)mk, 0u));
                    int base = 0;
                    if (first && rank == 0u) base = atomicAdd(&s_nseen, __popcll(mk));
                    base = __builtin_amdgcn_readlane(base, __builtin_ctzll(mk));
                    if (first) seen_list[base + (int)rank] = (u32)t;
                }
            }
        } else {
            for (int i = tid; i < hlen; i += NUC_BLOCK) {
                const int t = h[i];
                if (t < 0 || t >= V) atomicOr(a.status, 1);
                else if (r.penal) atomicOr(&bm[t >> 5], 1u << (t & 31));
            }
        }
        lds_barrier();
        {
            const int nseen = list_seen ? s_nseen : 0;
#pragma unroll
            for (int k = 0; k < NUC_SEEN; k++) {
                const int i = tid + k * NUC_BLOCK;
                seen_id[k] = i < nseen ? (int)seen_list[i] : -1;
            }
#pragma unroll
            for (int k = 0; k < NUC_SEEN; k++) seen_raw[k] = seen_id[k] >= 0 ? r.x[seen_id[k]] : 0.0f;
#pragma unroll
            for (int k = 0; k < NUC_SEEN; k++)
                seen_y[k] = seen_id[k] >= 0 ? penalise_seen(seen_raw[k], r.rep, r.counts, seen_id[k], r.freq, r.pres) : 0.0f;
        }
    };
    // every element of the row as f(id, penalised logit): the sweep, then the seen ids when the sweep masked them
    typename std::conditional<KEEP, NucKept<NUC_BLOCK>, NucNoFirst>::type kept;
    auto fill = [&]() {
        if constexpr (KEEP) return NucFill<NUC_BLOCK>{&kept};
        else return NucNoFirst();
    };
    auto sweep = [&](auto nt, auto f, auto pre, const auto &first) {
        nuc_foreach<NUC_BLOCK, decltype(nt)::value, NUC_BLOCK == 1024>(r, bm, f, pre, first);
        if (r.masked) {
#pragma unroll
            for (int k = 0; k < NUC_SEEN; k++)
                if (seen_id[k] >= 0) f(seen_id[k], seen_y[k]);
        }
    };
    // every element of the row as f(id, logit as stored): no penalty, no look at the history bitmap
    auto sweep_plain = [&](auto nt, auto f, const auto &first) {
        nuc_foreach<NUC_BLOCK, decltype(nt)::value, NUC_BLOCK == 1024, true>(r, bm, f, NucNoPre(), first);
    };
    typedef std::integral_constant<bool, false> Cached;             // the row is read again: ordinary loads
    typedef std::integral_constant<bool, true> Streamed;             // the row's last sweep: non-temporal loads

    BORN_STAMP(a, row, 1);
    // ---- sweep 1: maximum of the penalised logits, and about how far below it they reach
    {
        float mx = -INFINITY, mn = INFINITY;
        // (the smallest value only sizes the bins: every fourth id is looked at, spread over the whole row)
        sweep(Cached(), [&](int j, float y) {
            mx = fmaxf(mx, y);
            if ((j & 3) == 0) mn = fminf(mn, y > -3.402823466e+38f ? y : INFINITY);
        }, prologue, fill());
        mx = block_max_f32<NUC_BLOCK, true>(mx, &scr);
        mn = -block_max_f32<NUC_BLOCK, true>(-mn, &scr);
        r.m = uniform_f32(nuc_z(r, mx));
        r.degenerate = r.m == -INFINITY;                             // nothing finite: every d is 0 by definition
        const float zmin = mn < INFINITY ? nuc_z(r, mn) : r.m;
        const float span = r.degenerate ? 0.0f : r.m - zmin;         // >= 0
        // the bins cover the logits that can carry mass: the row's span, at most 32, at most the min-p bound
        r.range = uniform_f32(fminf(fminf(32.0f, span * 1.0001f + 1e-3f), r.dcut * 1.0001f + 1e-3f));
        r.sbin = uniform_f32((float)NUC_BINS / r.range);
        // sweeps 2 and 3: a value 200 below the maximum in z (no mass; outside every wanted range unless the last bin,
        // which takes everything beyond the span, is wanted: the gather then lists the constant once per seen id, with no
        // mass and ranked last, next to the id's real entry). A maximum that leaves no such value: penalties inside the sweeps.
        if (r.masked && fabsf(r.m) < 1e6f) r.skip = uniform_f32((r.m - 200.0f) * r.T);
        else r.masked = false;
        // The usual row (a maximum of ordinary size, a temperature whose division has the shortcut, no min-p bound, a history
        // short enough to be listed): sweeps 2 and 3 read the logits as stored, without the history bitmap, and what the
        // seen ids contribute is set right apart, see below.
        const float amx = fabsf(uniform_f32(mx)), am = fabsf(r.m);
        lin = !r.degenerate && am >= 0x1p-40f && am < 0x1p90f && amx < 0x1p90f && (r.T == 1.0f || r.rcp != 0.0f) &&
              r.dcut == 80.0f && (!r.penal || r.masked);
    }
    // In such a row the mass of a logit y needs no test of y at all. With x = z' - m, z' the three-instruction quotient
    // (y itself at temperature 1), the mass is that of exp(clamp(x, -87, 0)), and every kind of y comes out as specified:
    //   2^-100 <= |y| < 2^100  z' is the correctly rounded quotient, x = -d exactly;
    //   zeros and |y| < 2^-100  z' stays below 2^-78, half an ulp of m or less: x = -m, as with the exact z;
    //   -inf, NaN               x is -inf or a NaN (the quotient of -inf is inf - inf); the clamp (a median of three, which
    //                           returns the smallest operand when one is a NaN) gives -87: no mass;
    //   y <= -2^100             z' is -inf or within 2^-20 of the quotient, below -2^80: no mass;
    //   +inf, y >= 2^100        not in such a row (the maximum is below 2^90).
    // Beyond d = 80 the specified mass is 0, and so is trunc(exp(x) * 2^S) down to the clamp (S <= 61).  A seen id's
    // stored logit may exceed the penalised maximum: clamped to x = 0, some mass that the correction takes out again.
    const float nsbin = -r.sbin;
    const float scale32 = r.scale * 2.3283064365386963e-10f;
    // What lies beyond the bins (masked logits; all of a row far below one logit) goes to the last bin or one of the slots behind it by lane, which the scan adds to the last
    // bin: LDS atomics of 64 lanes on one bin are done one after the other.  us, all in the last bin and now, rows of which a mask leaves a tenth, then ordinary rows:
    // 8 x 50 257 53.2 21.4, 24.0 23.9; 64 x 32 000 37.7 17.2, 19.1 18.9; 128 x 152 064 146 51, 53 52; 512 x 8191 23.8 14.8, 15.1 15.4; in parts 32 x 128 256 36.6 27.0, 27.0 27.0.
    // (64 x 32 000 with 64 slots 17.1, with 8 17.7, 4 20.6.)
    const float beyond = (float)(NUC_BINS - 1 + (lane_id() & (NUC_BEYOND - 1)));
    auto lin_bin = [&](float x) { return (int)__builtin_amdgcn_fmed3f(x * nsbin, 0.0f, beyond); };   // (x from -87 to 0; the bins end at -32 or above)
    auto lin_z = [&](float y) { return r.T == 1.0f ? y : nuc_z_shortcut<ANY_T>(r, y); };
    auto lin_put = [&](float z, auto minus) {
        const float x = __builtin_amdgcn_fmed3f(z - r.m, -87.0f, 0.0f);
        const u64 q = qfix32(expneg_core(x), scale32);
        atomicAdd(&mass[lin_bin(x)], decltype(minus)::value ? 0ull - q : q);
    };
    typedef std::integral_constant<bool, false> Plus;
    typedef std::integral_constant<bool, true> Minus;

    BORN_STAMP(a, row, 2);
#if defined(BORN_NUC_STOP_AFTER) && BORN_NUC_STOP_AFTER == 1
    // (measurement builds only: the row ends after the named sweep, for per-sweep instruction counts; results are wrong)
    if (tid == 0) a.tokens[row] = __float_as_int(r.sbin) & 1;
    return;
#endif
    // ---- sweep 2: integer masses by bin
    if (lin) {
        if (r.penal) {
            // The histogram is a sum of integers modulo 2^64: the sweep adds every id's stored logit, so each seen id's stored
            // logit is taken out (by the same arithmetic, to the bit) and its penalised logit put in, here, in any order.
#pragma unroll
            for (int k = 0; k < NUC_SEEN; k++)
                if (seen_id[k] >= 0) {
                    lin_put(lin_z(seen_raw[k]), Minus());
                    lin_put(lin_z(seen_y[k]), Plus());
                }
        }
        if (a.mass_shift > 51) {                                     // (short rows)
            sweep_plain(Cached(), [&](int, float y) { lin_put(lin_z(y), Plus()); }, kept);
        } else {
            double start = mass_sum_start(a.mass_shift);
            mass_sum_begin(start);
            auto put = [&](float z) {
                const float x = __builtin_amdgcn_fmed3f(z - r.m, -87.0f, 0.0f);
                const u64 q = mass_of(expneg_core(x), start);
                atomicAdd(&mass[lin_bin(x)], q);
            };
            if (r.T == 1.0f) sweep_plain(Cached(), [&](int, float y) { put(y); }, kept);
            else sweep_plain(Cached(), [&](int, float y) { put(nuc_z_shortcut<ANY_T>(r, y)); }, kept);
            mass_sum_end(start);
        }
    } else if (r.T == 1.0f && !r.degenerate) {
        sweep(Cached(), [&](int, float y) {
            float z = y;                                             // a logit of ordinary magnitude is its own canonical form
            if (!nuc_ordinary(y)) {
                asm volatile("" ::: "memory");                       // (keeps this a branch: as selects it is paid by every logit)
                z = canon(y);
            }
            const float d = r.m - z;
            atomicAdd(&mass[nuc_bin(r, d)], qfix(expneg(d, r.dcut), r.scale));
        }, NucNoPre(), kept);
    } else if (r.rcp != 0.0f && !r.degenerate) {
        sweep(Cached(), [&](int, float y) {
            float z = nuc_z_shortcut<ANY_T>(r, y);
            if (!nuc_ordinary(y)) z = nuc_z(r, y);                   // zeros, masked (-inf) and other unusual logits: the division
            const float d = r.m - z;
            atomicAdd(&mass[nuc_bin(r, d)], qfix(expneg(d, r.dcut), r.scale));
        }, NucNoPre(), kept);
    } else {
        sweep(Cached(), [&](int, float y) {
            const float d = nuc_d(r, nuc_z(r, y));
            atomicAdd(&mass[nuc_bin(r, d)], qfix(expneg(d, r.dcut), r.scale));
        }, NucNoPre(), kept);
    }
    lds_barrier();
    BORN_STAMP(a, row, 3);
#if defined(BORN_NUC_STOP_AFTER) && BORN_NUC_STOP_AFTER == 2
    if (tid == 0) a.tokens[row] = (int)(mass[0] & 1ull);
    return;
#endif
    u64 Zk;
    {
        u64 v[NUC_PER], local = 0;
#pragma unroll
        for (int t = 0; t < NUC_PER; t++) {
            local += mass[tid * NUC_PER + t];
            v[t] = local;
        }
        static_assert(NUC_BEYOND <= NUC_WAVES * NUC_WCAP, "in the lists' storage");
        if (tid == NUC_BLOCK - 1) {
#pragma unroll
            for (int i = 0; i < NUC_BEYOND; i++) local += mass[NUC_BINS + i];
            v[NUC_PER - 1] = local;
        }
        const u64 excl = block_inclusive_scan_u64<NUC_BLOCK, true>(local, &scr, &Zk) - local;
#pragma unroll
        for (int t = 0; t < NUC_PER; t++) mass[tid * NUC_PER + t] = v[t] + excl;
    }
    lds_barrier();
    const u64 *cum = mass;

    // ---- the bins to gather: the top-p cut's, w0, and those that the draw may fall into, w1 to w2.  The mass of the nucleus lies in
    // [tp, cum[w0]], which bounds the draw's target.  All of w1 .. w2 are few logits: what lies strictly between them adds up to at most the
    // mass of bin w0, and each of its logits has at least the mass of any in w0 (w2 <= w0), so there are no more of them than w0 holds.
    // (Before, up to two such bins, else the cut's alone and two more sweeps of the row for a draw elsewhere.  us, then and now: 96 x 100 003, settings
    // per row, 78 and 49 (50 where every row's draw was in those two bins); 256 x 128 256 of twenty likely tokens, top-p 0.9, 131 and 82; 100 x 300 23.6 and 12.1.)
    const bool cut = cfg_p < 1.0f;
    u64 tp = Zk;
    int w0, w1, w2;
    if (cut) {
        tp = top_p_target(cfg_p, Zk);
        w0 = nuc_first_reaching(cum, tp);
        const u64 hi = cum[w0] < Zk ? cum[w0] : Zk;
        w1 = nuc_first_reaching(cum, draw_target(u, tp));
        w2 = nuc_first_reaching(cum, draw_target(u, hi));
    } else {
        w0 = w1 = w2 = nuc_first_reaching(cum, draw_target(u, Zk));
    }

    BORN_STAMP(a, row, 4);
    // ---- sweep 3: stage the logits inside the wanted bins' ranges, then classify them exactly
    bool listed;
    {
        // The cut's bin, and above it (w2 <= w0) the draw's; one interval where the two meet.
        float lo0, hi0, lo1, hi1, lo2, hi2;
        nuc_range(r, w0, lo0, hi0);
        nuc_range(r, w1, lo1, hi1);
        nuc_range(r, w2, lo2, hi2);
        lo1 = lo2;
        const bool one = !(lo1 > hi0);
        if (one) hi0 = fmaxf(hi0, hi1);
        const NucList staged{stage + wave_id() * NUC_WCAP, &s_wcount[wave_id()]};
        staged.clear();
        auto append = [&](u64 mk, float y, int j) { staged.template append<NUC_WCAP>(mk, y, j); };
        auto in_one = [&](float y) { return nuc_within(y, lo0, hi0); };
        auto in_either = [&](float y) { return nuc_within(y, lo0, hi0) | nuc_within(y, lo1, hi1); };
        auto sweep_few = [&](auto wanted) {
            nuc_foreach4<NUC_BLOCK, true, NUC_BLOCK == 1024, true>(r, bm, [&](int j, const float (&y)[4]) { staged.template append4<NUC_WCAP>(wanted, y, j); },
                                                                   [&](int j, float y) { append(wanted(y), y, j); }, NucNoPre(), kept);
        };
        if (lin) {
            // (the stored logits; a seen id's stored logit that passes is dropped below, its penalised logit is offered
            // here under the id with the top bit set)
            if (one) sweep_few(in_one);
            else sweep_few(in_either);
            if (r.penal) {
#pragma unroll
                for (int k = 0; k < NUC_SEEN; k++)
                    if (seen_id[k] >= 0) {
                        append(in_either(seen_y[k]), seen_y[k], (int)((u32)seen_id[k] | 0x80000000u));
                    }
            }
        } else if (one) {
            sweep(Streamed(), [&](int j, float y) { append(in_one(y), y, j); }, NucNoPre(), kept);
        } else {
            sweep(Streamed(), [&](int j, float y) { append(in_either(y), y, j); }, NucNoPre(), kept);
        }
        const u32 count = staged.size();
        if (count > (u32)NUC_WCAP && lane_id() == 0) s_over = 1;
        const int cw = (int)min(count, (u32)NUC_WCAP);
        auto classify = [&]() {
            for (int e0 = 0; e0 < cw; e0 += WAVE) {
                const int e = e0 + lane_id();
                bool take = false;
                u64 key = 0ull, qs = 0ull;
                if (e < cw) {
                    uint2 c = staged.at[e];
                    bool stale = false;                                  // a seen id's stored logit
                    if (lin && r.penal) {
                        if (c.y & 0x80000000u) c.y &= 0x7FFFFFFFu;
                        else stale = (bm[c.y >> 5] >> (c.y & 31)) & 1u;
                    }
                    const float z = nuc_z(r, __uint_as_float(c.x));
                    const float d = nuc_d(r, z);
                    const int b = nuc_bin(r, d);
                    const int slot = stale ? -1 : b == w0 ? 0 : b >= w1 && b <= w2 ? 1 : -1;
                    if (slot >= 0) {
                        take = true;
                        key = make_key64(z, (int)c.y);
                        qs = qfix(expneg(d, r.dcut), r.scale) | ((u64)slot << 62);
                    }
                }
                const u64 mk = __ballot(take);
                if (mk) {
                    int base = 0;
                    if (lane_id() == 0) base = atomicAdd(&s_n, __popcll(mk));
                    base = __builtin_amdgcn_readfirstlane(base);
                    if (take) {
                        const int pos = base + (int)__builtin_amdgcn_mbcnt_hi((u32)(mk >> 32), __builtin_amdgcn_mbcnt_lo((u32)mk, 0u));
                        if (pos < NUC_CAP) {
                            fkey[pos] = key;
                            fq[pos] = qs;
                        }
                    }
                }
            }
        };
        classify();
        __syncthreads();
        listed = !s_over && s_n <= NUC_CAP;                          // the wanted bins fit the lists
        if (!listed && !s_over && w1 < w0) {
            // (uniform) Equal logits may make w1 and w2 themselves as full as w0.  Where w0's alone fit, they are listed, and the draw's bin is left to the descent
            // (us, both by the descent and so: logits of steps of 0.07, 200 x 50 257 153 98, 32 x 32 000 131 90, 200 x 128 256 244 155)
            w1 = w2 = w0;
            __syncthreads();
            if (tid == 0) s_n = 0;
            __syncthreads();
            classify();
            __syncthreads();
            listed = s_n <= NUC_CAP;
        }
    }
    BORN_STAMP(a, row, 5);
    const int n = listed ? s_n : 0;
    const int n4 = (n + 3) & ~3;                                     // the list padded to whole groups of four ..
    if (tid >= n && tid < n4) {
        fkey[tid] = 0ull;                                            // .. with entries of no slot and no mass
        fq[tid] = 3ull << 62;
    }
    __syncthreads();

    // ---- cumulative mass of every listed entry within its bin, in rank order.  The bins' value ranges are disjoint, so
    // the rank order of the whole list goes bin by bin: an entry counts the keys above its own (all distinct: the id is
    // part of the key) and moves to that place; one scan of the masses in that order gives every entry the mass at and
    // above it, and where a bin begins the scan holds what the bins listed before it add up to.  128 buckets for the range of either slot (the draw's bins lie above
    // the cut's): an entry counts the keys of its own bucket only.  Bound by the chain of LDS round trips.  (Against the whole list, then the
    // targets by an LDS maximum and five barriers each: the resolve of the slowest row of 96 x 100 003 took 10 us, 3.8 so, of 1024 x 152 064 7.8 and 3.0;
    // lists of 33 to 128 entries, summed directly before, 5.8 and 3.7.)
    u64 mykey = 0ull, mine = 0ull, q = 0ull;                         // its own mass, and the mass at and above it in its bin
    int myslot = -1;
    if (n <= NUC_DIRECT) {
        // (a short list: every entry sums the masses of its bin's entries at and above it; no barrier, no scan)
        if (tid < n) {
            mykey = fkey[tid];
            myslot = (int)(fq[tid] >> 62);
            q = fq[tid] & 0x3FFFFFFFFFFFFFFFull;
            const ulonglong2 *k2 = reinterpret_cast<const ulonglong2 *>(fkey), *q2 = reinterpret_cast<const ulonglong2 *>(fq);
            for (int j = 0; j < n4; j += 4) {
                const ulonglong2 ka = k2[j >> 1], kb = k2[(j >> 1) + 1], qa = q2[j >> 1], qb = q2[(j >> 1) + 1];
                const u64 ks[4] = {ka.x, ka.y, kb.x, kb.y}, qs[4] = {qa.x, qa.y, qb.x, qb.y};
#pragma unroll
                for (int t = 0; t < 4; t++)
                    if ((int)(qs[t] >> 62) == myslot && ks[t] >= mykey) mine += qs[t] & 0x3FFFFFFFFFFFFFFFull;
            }
        }
    } else {
        u64 *const skey = reinterpret_cast<u64 *>(stage), *const sq = skey + NUC_CAP;       // the staging lists are spent
        u32 *const count = reinterpret_cast<u32 *>(sq + NUC_CAP), *const at = count + 256;
        static_assert(2 * NUC_CAP + 256 <= NUC_WAVES * NUC_WCAP, "the ordered entries and the buckets fit the staging lists' storage");
        if (tid < 256) count[tid] = 0u;
        if (tid < 2) {
            s_top[tid] = 0u;
            s_low[tid] = ~0u;
        }
        const u64 key = tid < n ? fkey[tid] : 0ull, kq = tid < n ? fq[tid] : 0ull;
        const u32 z = (u32)(key >> 32);
        const int in_slot = (int)(kq >> 62);
        lds_barrier();
        if ((tid & ~(WAVE - 1)) < n) {                               // wave-uniform
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const bool its = tid < n && in_slot == t;
                const u32 most = wave_max_u32(its ? z : 0u), least = wave_min_u32(its ? z : ~0u);
                if (lane_id() == 0) {
                    atomicMax(&s_top[t], most);
                    atomicMin(&s_low[t], least);
                }
            }
        }
        lds_barrier();
        u32 bucket = 0u, pos = 0u;
        if (tid < n) {
            const u32 range = s_top[in_slot] - s_low[in_slot];
            const int sh = max(0, 25 - (int)__clz(range));           // (range >> sh) < 128
            bucket = (in_slot ? 0u : 128u) + ((s_top[in_slot] - z) >> sh);
            pos = atomicAdd(&count[bucket], 1u);
        }
        lds_barrier();
        if (tid < WAVE) {
            const uint4 c = reinterpret_cast<const uint4 *>(count)[tid];
            const u32 four = c.x + c.y + c.z + c.w, ex = wave_inclusive_scan_u32(four) - four;
            reinterpret_cast<uint4 *>(at)[tid] = make_uint4(ex, ex + c.x, ex + c.x + c.y, ex + c.x + c.y + c.z);
        }
        lds_barrier();
        const u32 begin = tid < n ? at[bucket] : 0u;
        if (tid < n) fkey[begin + pos] = key;                        // (by bucket; the keys that pad the list stay behind them)
        lds_barrier();
        if (tid < n) {
            // four keys a turn, from a whole group of four on: those of earlier buckets count, those of later ones do not
            const u32 end = begin + count[bucket];
            u32 j = begin & ~3u, rank = j;
            const ulonglong2 *k2 = reinterpret_cast<const ulonglong2 *>(fkey);
            for (; j < end; j += 4) {
                const ulonglong2 ka = k2[j >> 1], kb = k2[(j >> 1) + 1];
                rank += (u32)(ka.x > key) + (u32)(ka.y > key) + (u32)(kb.x > key) + (u32)(kb.y > key);
            }
            skey[rank] = key;
            sq[rank] = kq;
        }
        __syncthreads();
        if (tid < n) {
            mykey = skey[tid];
            const u64 w = sq[tid];
            myslot = (int)(w >> 62);
            q = w & 0x3FFFFFFFFFFFFFFFull;
        }
        u64 listed_mass;
        const u64 incl = block_inclusive_scan_u64<NUC_BLOCK>(q, &scr, &listed_mass);
        if (tid < n && (tid == 0 || (int)(sq[tid - 1] >> 62) != myslot)) s_slot0[myslot] = incl - q;
        __syncthreads();
        if (tid < n) mine = incl - s_slot0[myslot];
    }
    // ---- the cut, then the draw: each is the first element in rank order of one bin at which the cumulative
    // mass reaches a target.  Listed bins are resolved from `mine`; a bin that is not (heavy ties: the lists overflowed, or the cut's alone were gathered) by a radix
    // descent over its rank keys, 11 bits per sweep, until its bucket fits the list.
    r.masked = false;                                                // (the sweeps of a radix descent apply the penalties themselves)
    u64 Zp = Zk, tokkey = 0ull;
    u64 *const smass = reinterpret_cast<u64 *>(stage);               // [2048] sub-histogram of masses
    u32 *const scnt = reinterpret_cast<u32 *>(fkey);                 // [2048] and of counts
    for (int phase = cut ? 0 : 1; phase < 2; phase++) {
        const u64 target = phase == 0 ? tp : draw_target(u, Zp);
        const int b = phase == 0 ? w0 : nuc_first_reaching(cum, target);
        u64 base = b ? cum[b - 1] : 0ull;
        const int slot = !listed ? -1 : b == w0 ? 0 : b >= w1 && b <= w2 ? 1 : -1;
        if (slot == 1) base = w1 ? cum[w1 - 1] : 0ull;               // (listed from w1 on)
        if (slot < 0) {
            __syncthreads();                                         // (the lists are overwritten)
            u64 prefix = 0ull;
            int plen = 0;
            for (;;) {
                const int db = min(11, 64 - plen), nsb = 1 << db;
                for (int i = tid; i < nsb; i += NUC_BLOCK) {
                    smass[i] = 0ull;
                    scnt[i] = 0u;
                }
                __syncthreads();
                {
                    const u64 pf = prefix;
                    const int pl = plen;
                    nuc_foreach<NUC_BLOCK>(r, bm, [&](int j, float y) {
                        const float z = nuc_z(r, y);
                        const float d = nuc_d(r, z);
                        if (nuc_bin(r, d) != b) return;
                        const u64 key = make_key64(z, j);
                        if (pl > 0 && (key >> (64 - pl)) != pf) return;
                        const int idx = nsb - 1 - (int)((key >> (64 - pl - db)) & (u64)(nsb - 1));   // larger keys first
                        atomicAdd(&smass[idx], qfix(expneg(d, r.dcut), r.scale));
                        atomicAdd(&scnt[idx], 1u);
                    });
                }
                __syncthreads();
                {
                    // inclusive scan over nsb <= 2048 sub-bins, NUC_SUB consecutive ones per thread
                    u64 c[NUC_SUB], sum = 0ull;
#pragma unroll
                    for (int t = 0; t < NUC_SUB; t++) {
                        const int i = NUC_SUB * tid + t;
                        sum += i < nsb ? smass[i] : 0ull;
                        c[t] = sum;
                    }
                    u64 tot;
                    const u64 excl = block_inclusive_scan_u64<NUC_BLOCK>(sum, &scr, &tot) - sum;
#pragma unroll
                    for (int t = 0; t < NUC_SUB; t++) {
                        const int i = NUC_SUB * tid + t;
                        if (i < nsb) smass[i] = excl + c[t];
                    }
                }
                __syncthreads();
                int lo = 0, hi = nsb - 1;                            // first sub-bin at which base + cumulative reaches target
                while (lo < hi) {
                    const int mid = (lo + hi) >> 1;
                    if (base + smass[mid] >= target) hi = mid; else lo = mid + 1;
                }
                const u32 cntb = scnt[lo];
                base += lo ? smass[lo - 1] : 0ull;
                prefix = (prefix << db) | (u64)(nsb - 1 - lo);
                plen += db;
                __syncthreads();
                if (cntb <= (u32)NUC_CAP || plen == 64) break;
            }
            // list the bucket and sum within it
            if (tid == 0) s_n = 0;
            __syncthreads();
            {
                const u64 pf = prefix;
                const int pl = plen;
                nuc_foreach<NUC_BLOCK>(r, bm, [&](int j, float y) {
                    const float z = nuc_z(r, y);
                    const float d = nuc_d(r, z);
                    if (nuc_bin(r, d) != b) return;
                    const u64 key = make_key64(z, j);
                    if (pl < 64 ? (key >> (64 - pl)) != pf : key != pf) return;
                    const int pos = atomicAdd(&s_n, 1);
                    if (pos < NUC_CAP) {
                        fkey[pos] = key;
                        fq[pos] = qfix(expneg(d, r.dcut), r.scale);          // slot 0
                    }
                });
            }
            __syncthreads();
            const int nb = min(s_n, NUC_CAP);
            mykey = 0ull;
            mine = 0ull;
            myslot = -1;
            if (tid < nb) {
                mykey = fkey[tid];
                q = fq[tid];
                myslot = 0;
                for (int j = 0; j < nb; j++)
                    if (fkey[j] >= mykey) mine += fq[j];
            }
            __syncthreads();
        }
        // the first entry in rank order at which base + cumulative reaches the target: the one whose own mass crosses it
        const int sl = slot < 0 ? 0 : slot;
        if (myslot == sl && base + mine >= target && base + (mine - q) < target) {
            s_win[phase] = mykey;
            s_mass[phase] = base + mine;
        }
        __syncthreads();
        const u64 win = s_win[phase];
        if (phase == 0) Zp = s_mass[0];
        else tokkey = win;
        if (win == 0ull) break;                                      // inconsistent histogram: cannot happen
    }
    BORN_STAMP(a, row, 6);
    if (tid == 0) {
        if (tokkey == 0ull) {
            atomicOr(a.status, 4);                                   // internal inconsistency, reported by the status call
            a.tokens[row] = 0;
            if (a.probs) a.probs[row] = 0.0f;
        } else {
            a.tokens[row] = key64_id(tokkey);
            if (a.probs) a.probs[row] = prob_of(emass(key64_z(tokkey), r.m, r.dcut), Zp, a.mass_shift);
        }
        if (a.nuc_len) a.nuc_len[row] = -1;                          // the nucleus listing is only produced for small top-k
        count_row(a.counters, row, listed ? 2 : 1);
        if (!listed) count_row(a.counters, row, 2);
    }
    BORN_STAMP(a, row, 7);
}

// Rows that start at any four bytes are read by 128-bit loads from this length on: a shorter one leaves most lanes without such a
// load and reads its ragged end after it, a second round trip to memory (22 x 101: 11.6 us one logit at a time, 12.8 by 128-bit loads;
// 600 x 1001 27.1 and 28.2; 2039 27.1 and 26.0; 8191 35.8 and 28.1).
constexpr int NUC_LOADS4_FROM = 1536;
static inline int row_blocks(const SampleArgs &a) { return a.V >= NUC_LOADS4_FROM || rows_aligned(a.logits, a.row_stride) ? a.V >> 2 : 0; }

}  // namespace born
