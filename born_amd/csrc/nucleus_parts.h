// Rows without a top-k cut, each by several workgroups: included at the end of nucleus_row.hip, whose row visitor, bins and
// arithmetic it uses.
//
// A workgroup per row leaves most of the device idle where the batch has fewer rows than half the CUs, and a row's three sweeps are
// then the time of all (sweep 2's arithmetic, 28 vector instructions per logit on one CU, the larger part of it).  Here a row is
// cut into parts of whole 128-byte lines, a workgroup to each, and the sweeps are launches: what a part finds is small,
// and the end of a launch is what makes it known to the others.
//   max      maximum and smallest finite value of the part's penalised logits.
//   masses   the masses of the part by bin, as in the one-workgroup kernel, and their sums over runs of 64 bins.
//   gather   every part finds the wanted bins for itself: the runs' sums of all parts first, then the bins of the
//            runs that hold a target (at most three: 1.5 KiB a part instead of the 32 KiB of all bins), and lists its own logits of them.
//   draw     a workgroup per row puts the lists in rank order, finds the cut and draws.
// Rows that are not "usual" (the same test as in the one-workgroup kernel, but any temperature: ANY_T) and lists that overflow
// are the last launch's, which runs the one-workgroup body for them.  The bits are the same on every route: integer sums, and exact rank keys.
#include "nucleus_plan.h"

namespace born {

constexpr int PARTS_BLOCK = 1024;
constexpr int PARTS_RUN = WAVE, PARTS_RUNS = NUC_BINS / PARTS_RUN;   // runs of bins
constexpr int PARTS_LIST = 512;               // gathered entries of a part
constexpr int PARTS_CAP = PARTS_BLOCK;        // of a row
constexpr int PARTS_SEEN = 4;                 // seen ids a thread keeps: histories of at most 4096 tokens
constexpr int PARTS_TOTAL = 256;              // of a batch, at most
static_assert(PARTS_RUNS == WAVE, "one lane per run, one per bin of a run");
static_assert(PARTS_ROW_MAX * PARTS_RUN <= 2 * PARTS_BLOCK && PARTS_ROW_MAX <= WAVE, "sums over parts");

struct PartsArgs {
    int parts, len;                           // of a row; logits of a part (the last one: what is left)
    u64 *bins;                                // [row][part][NUC_BINS]
    u64 *runs;                                // [row][part][PARTS_RUNS]
    ulonglong2 *list;                         // [row][part][PARTS_LIST] rank key, mass | slot << 62
    float2 *ends;                             // [row][part] maximum, smallest finite value
    u32 *count;                               // [row][part] gathered entries; above PARTS_LIST: lists overflowed
    struct PartsRow *rows;                    // [row]
};

struct PartSeen {
    int id[PARTS_SEEN];                       // within the part, each once; -1: none
    float raw[PARTS_SEEN], y[PARTS_SEEN];
};

// The part as a row of its own (ids from 0), and the ids of the row's history that lie in it.
struct Part {
    NucRow r;
    int lo;
    const int *h;
    int hlen;
};
__device__ __forceinline__ Part part_of(const SampleArgs &a, const PartsArgs &pa) {
    Part p;
    const int row = blockIdx.x;
    p.lo = (int)blockIdx.y * pa.len;
    NucRow &r = p.r;
    r.x = a.logits + (long long)row * a.row_stride + p.lo;
    r.V = min(pa.len, a.V - p.lo);
    r.n4 = r.V >> 2;
    r.T = a.T;
    r.rcp = nuc_reciprocal(a.T);
    r.rep = a.rep;
    r.scale = mass_scale(a.mass_shift);
    r.dcut = a.dcut;
    r.counts = nullptr;
    r.freq = r.pres = 0.0f;
    r.degenerate = false;
    r.m = r.range = r.sbin = 0.0f;
    p.hlen = a.history ? min((int)(a.hist_len ? a.hist_len[row] : (int)a.hist_stride), (int)a.hist_stride) : 0;
    p.h = a.history + (long long)row * a.hist_stride;
    r.penal = a.rep != 1.0f && p.hlen > 0;
    r.masked = r.penal;
    r.skip = -INFINITY;
    return p;
}
// Sets the part's bits of the history bitmap and lists its seen ids, each once; every thread keeps up to PARTS_SEEN of them.
// bm: one bit per id of the part; list: PARTS_SEEN * PARTS_BLOCK words.  Barriers that order LDS traffic only.
__device__ __forceinline__ void part_history(const SampleArgs &a, const Part &p, bool report, u32 *bm, u32 *list, int *s_n, PartSeen &seen) {
    const int tid = threadIdx.x;
    const NucRow &r = p.r;
    if (r.penal)
        for (int i = tid; i < ((r.V + 31) >> 5); i += PARTS_BLOCK) bm[i] = 0u;
    if (tid == 0) *s_n = 0;
    lds_barrier();
    if (r.penal || report) {
        int hv[PARTS_SEEN];
#pragma unroll
        for (int k = 0; k < PARTS_SEEN; k++) {
            const int i = tid + k * PARTS_BLOCK;
            hv[k] = i < p.hlen ? p.h[i] : -2;
        }
#pragma unroll
        for (int k = 0; k < PARTS_SEEN; k++) {
            const int i = tid + k * PARTS_BLOCK, t = hv[k] >= p.lo ? hv[k] - p.lo : -1;
            if (report && i < p.hlen && (hv[k] < 0 || hv[k] >= a.V)) atomicOr(a.status, 1);
            bool first = false;
            if (r.penal && t >= 0 && t < r.V) {
                const u32 bit = 1u << (t & 31);
                first = !(atomicOr(&bm[t >> 5], bit) & bit);
            }
            const u64 mk = __ballot(first);
            if (mk) {
                const u32 rank = __builtin_amdgcn_mbcnt_hi((u32)(mk >> 32), __builtin_amdgcn_mbcnt_lo((u32)mk, 0u));
                int base = 0;
                if (first && rank == 0u) base = atomicAdd(s_n, __popcll(mk));
                base = __builtin_amdgcn_readlane(base, __builtin_ctzll(mk));
                if (first) list[base + (int)rank] = (u32)t;
            }
        }
    }
    lds_barrier();
    const int n = *s_n;
#pragma unroll
    for (int k = 0; k < PARTS_SEEN; k++) {
        const int i = tid + k * PARTS_BLOCK;
        seen.id[k] = i < n ? (int)list[i] : -1;
    }
#pragma unroll
    for (int k = 0; k < PARTS_SEEN; k++) seen.raw[k] = seen.id[k] >= 0 ? r.x[seen.id[k]] : 0.0f;
#pragma unroll
    for (int k = 0; k < PARTS_SEEN; k++) seen.y[k] = seen.id[k] >= 0 ? penalise(seen.raw[k], r.rep) : 0.0f;
}
// The row's maximum and bins from what its parts found; whether the row is usual (nucleus_row_body says of what that consists).
__device__ __forceinline__ bool part_bins(NucRow &r, const PartsArgs &pa) {
    const int l = lane_id();
    float2 e = make_float2(-INFINITY, INFINITY);
    if (l < pa.parts) e = pa.ends[(long long)blockIdx.x * pa.parts + l];
    const float mx = wave_max_f32(e.x), mn = -wave_max_f32(-e.y);
    r.m = uniform_f32(nuc_z(r, mx));
    r.degenerate = r.m == -INFINITY;
    const float zmin = mn < INFINITY ? nuc_z(r, mn) : r.m;
    const float span = r.degenerate ? 0.0f : r.m - zmin;
    r.range = uniform_f32(fminf(32.0f, span * 1.0001f + 1e-3f));
    r.sbin = uniform_f32((float)NUC_BINS / r.range);
    const float amx = fabsf(uniform_f32(mx)), am = fabsf(r.m);
    return !r.degenerate && am >= 0x1p-40f && am < 0x1p90f && amx < 0x1p90f && (r.T == 1.0f || r.rcp != 0.0f) && r.dcut == 80.0f;
}
__device__ __forceinline__ float part_z(const NucRow &r, float y) { return r.T == 1.0f ? y : nuc_z_shortcut<true>(r, y); }

__global__ __launch_bounds__(PARTS_BLOCK, 4) void nucleus_parts_max_kernel(SampleArgs a, PartsArgs pa) {
    extern __shared__ __align__(16) u64 nuc_dyn[];                   // seen ids, then the bitmap
    __shared__ BlockScratch scr;
    __shared__ int s_n;
    u32 *const list = reinterpret_cast<u32 *>(nuc_dyn), *const bm = list + PARTS_SEEN * PARTS_BLOCK;
    const Part p = part_of(a, pa);
    PartSeen seen;
    float mx = -INFINITY, mn = INFINITY;
    auto look = [&](int j, float y) {
        mx = fmaxf(mx, y);
        if ((j & 3) == 0) mn = fminf(mn, y > -3.402823466e+38f ? y : INFINITY);
    };
    nuc_foreach<PARTS_BLOCK, false, true>(p.r, bm, look, [&]() { part_history(a, p, blockIdx.y == 0, bm, list, &s_n, seen); });
    if (p.r.penal) {
#pragma unroll
        for (int k = 0; k < PARTS_SEEN; k++)
            if (seen.id[k] >= 0) look(seen.id[k], seen.y[k]);
    }
    mx = block_max_f32<PARTS_BLOCK>(mx, &scr);
    mn = -block_max_f32<PARTS_BLOCK>(-mn, &scr);
    if (threadIdx.x == 0) pa.ends[(long long)blockIdx.x * pa.parts + blockIdx.y] = make_float2(mx, mn);
}

__global__ __launch_bounds__(PARTS_BLOCK, 4) void nucleus_parts_masses_kernel(SampleArgs a, PartsArgs pa) {
    extern __shared__ __align__(16) u64 nuc_dyn[];                   // bins and the slots beyond them, seen ids, the bitmap
    __shared__ int s_n;
    u64 *const mass = nuc_dyn;
    u32 *const list = reinterpret_cast<u32 *>(nuc_dyn + NUC_BINS + NUC_BEYOND), *const bm = list + PARTS_SEEN * PARTS_BLOCK;
    const int tid = threadIdx.x;
    Part p = part_of(a, pa);
    if (!part_bins(p.r, pa)) return;                                 // workgroup-uniform
    const NucRow &r = p.r;
    const float scale32 = r.scale * 2.3283064365386963e-10f, nsbin = -r.sbin;
    const float beyond = (float)(NUC_BINS - 1 + (lane_id() & (NUC_BEYOND - 1)));          // (see nucleus_row_body)
    auto bin = [&](float x) { return (int)__builtin_amdgcn_fmed3f(x * nsbin, 0.0f, beyond); };
    auto put = [&](float z, bool minus) {
        const float x = __builtin_amdgcn_fmed3f(z - r.m, -87.0f, 0.0f);
        const u64 q = qfix32(expneg_core(x), scale32);
        atomicAdd(&mass[bin(x)], minus ? 0ull - q : q);
    };
    auto prologue = [&]() {
        for (int i = tid; i < NUC_BINS + NUC_BEYOND; i += PARTS_BLOCK) mass[i] = 0ull;
        if (r.penal) {
            PartSeen seen;
            part_history(a, p, false, bm, list, &s_n, seen);         // (its barriers stand behind the bins' zeros)
#pragma unroll
            for (int k = 0; k < PARTS_SEEN; k++)
                if (seen.id[k] >= 0) {                               // a seen id's stored logit out, its penalised logit in
                    put(part_z(r, seen.raw[k]), true);
                    put(part_z(r, seen.y[k]), false);
                }
        } else {
            lds_barrier();
        }
    };
    static_assert(PARTS_SPARED >= 1024, "mass_of's shift");
    double start = mass_sum_start(a.mass_shift);
    mass_sum_begin(start);
    auto add = [&](float z) {
        const float x = __builtin_amdgcn_fmed3f(z - r.m, -87.0f, 0.0f);
        const u64 q = mass_of(expneg_core(x), start);
        atomicAdd(&mass[bin(x)], q);
    };
    if (r.T == 1.0f) nuc_foreach<PARTS_BLOCK, false, true, true>(r, bm, [&](int, float y) { add(y); }, prologue);
    else nuc_foreach<PARTS_BLOCK, false, true, true>(r, bm, [&](int, float y) { add(nuc_z_shortcut<true>(r, y)); }, prologue);
    mass_sum_end(start);
    __syncthreads();
    const long long part = (long long)blockIdx.x * pa.parts + blockIdx.y;
    u64 *const out = pa.bins + part * NUC_BINS, *const sums = pa.runs + part * PARTS_RUNS;
    u64 more = 0ull;
    if (tid == PARTS_BLOCK - 1) {                                    // (the last bin's)
#pragma unroll
        for (int i = 0; i < NUC_BEYOND; i++) more += mass[NUC_BINS + i];
    }
    for (int i = tid; i < NUC_BINS; i += PARTS_BLOCK) {              // a wave: a run of bins
        const u64 q = mass[i] + (i == NUC_BINS - 1 ? more : 0ull);
        out[i] = q;
        const u64 s = wave_inclusive_scan_u64(q);
        if (lane_id() == WAVE - 1) sums[i / PARTS_RUN] = s;
    }
}

// A wanted bin: the first at which the mass from the row's maximum down reaches a target.
struct PartsBin {
    int bin;
    u64 before, upto;                         // the mass above the bin; and with it
};

// What the parts' gather knows of its row and the finish needs.
struct PartsRow {
    u64 tp, Zk;
    u64 before[2];                            // the mass above the listed bins: those of the cut (slot 0), those of the draw (slot 1)
    float m;
    int draw, alone;                          // the draw's slot; the row is left to the one-workgroup body
};

__global__ __launch_bounds__(PARTS_BLOCK, 4) void nucleus_parts_gather_kernel(SampleArgs a, PartsArgs pa) {
    extern __shared__ __align__(16) u64 nuc_dyn[];                   // staged logits, seen ids, the bitmap
    constexpr int WAVES = PARTS_BLOCK / WAVE, WCAP = NucGeom<PARTS_BLOCK>::WCAP;
    __shared__ u64 s_runs[PARTS_RUNS], s_bins[3][PARTS_RUN];
    __shared__ u32 s_wcount[WAVES];
    __shared__ int s_n, s_over;
    const int tid = threadIdx.x, row = blockIdx.x, l = lane_id();
    const bool tells = blockIdx.y == 0 && tid == 0;
    Part p = part_of(a, pa);
    const bool usual = part_bins(p.r, pa);
    const NucRow &r = p.r;
    if (!usual) {                                                    // (the same in every part)
        if (tells) pa.rows[row].alone = 1;
        return;
    }
    // (the first of the part's logits, for its sweep: in flight while the wanted bins are found)
    nuc_f32x4 first[NucGeom<PARTS_BLOCK>::U];
    nuc_request_first<PARTS_BLOCK, true>(r, first);
    const float u = a.uniforms ? a.uniforms[row] : uniform_of(a.seed, a.step, (u64)row);
    const u64 *const runs = pa.runs + (long long)row * pa.parts * PARTS_RUNS, *const bins = pa.bins + (long long)row * pa.parts * NUC_BINS;

    if (tid < PARTS_RUNS) {
        s_runs[tid] = 0ull;
        s_bins[0][tid] = s_bins[1][tid] = s_bins[2][tid] = 0ull;
    }
    if (tid == 0) s_over = 0;
    lds_barrier();
    for (int i = tid; i < pa.parts * PARTS_RUNS; i += PARTS_BLOCK) atomicAdd(&s_runs[i & (PARTS_RUNS - 1)], runs[i]);
    lds_barrier();
    const u64 run_mass = s_runs[l], run_upto = wave_inclusive_scan_u64(run_mass);   // (every wave for itself)
    const u64 Zk = shfl_u64(run_upto, WAVE - 1);
    auto run_of = [&](u64 target) {
        const u64 b = __ballot(run_upto >= target);
        return b ? __builtin_ctzll(b) : WAVE - 1;
    };
    auto fetch = [&](int run, u64 *to) {                             // the run's bins, summed over the parts
        for (int i = tid; i < pa.parts * PARTS_RUN; i += PARTS_BLOCK)
            atomicAdd(&to[i & (PARTS_RUN - 1)], bins[(long long)(i / PARTS_RUN) * NUC_BINS + run * PARTS_RUN + (i & (PARTS_RUN - 1))]);
    };
    auto bin_of = [&](u64 target, int run, const u64 *from) {
        const u64 base = shfl_u64(run_upto, run) - shfl_u64(run_mass, run), q = from[l], upto = base + wave_inclusive_scan_u64(q);
        const u64 b = __ballot(upto >= target);
        const int at = b ? __builtin_ctzll(b) : WAVE - 1;
        PartsBin w;
        w.bin = run * PARTS_RUN + at;
        w.upto = shfl_u64(upto, at);
        w.before = w.upto - shfl_u64(q, at);
        return w;
    };

    // The cut's bin, and the bins the draw may fall into: the nucleus mass lies between tp and the mass down to the end of the cut's bin, and
    // the draw's target grows with it.  Where those reach the cut's bin both are one range of bins.
    const bool cut = a.top_p < 1.0f;
    u64 tp = Zk;
    PartsBin w0, w1, w2;
    if (cut) {
        tp = top_p_target(a.top_p, Zk);
        const int c0 = run_of(tp);
        fetch(c0, s_bins[0]);
        lds_barrier();
        w0 = bin_of(tp, c0, s_bins[0]);
        const u64 hi = w0.upto < Zk ? w0.upto : Zk, t1 = draw_target(u, tp), t2 = draw_target(u, hi);
        const int c1 = run_of(t1), c2 = run_of(t2);
        fetch(c1, s_bins[1]);
        if (c2 != c1) fetch(c2, s_bins[2]);
        lds_barrier();
        w1 = bin_of(t1, c1, s_bins[1]);
        w2 = bin_of(t2, c2, c2 != c1 ? s_bins[2] : s_bins[1]);
    } else {
        const u64 t = draw_target(u, Zk);
        const int c = run_of(t);
        fetch(c, s_bins[0]);
        lds_barrier();
        w0 = w1 = w2 = bin_of(t, c, s_bins[0]);
    }
    const bool joined = w2.bin >= w0.bin;

    // ---- the part's logits of the wanted bins: staged by value ranges that can only over-select, then classified
    uint2 *const stage = reinterpret_cast<uint2 *>(nuc_dyn);                      // [WAVES][WCAP]
    u32 *const seen_list = reinterpret_cast<u32 *>(nuc_dyn + WAVES * WCAP), *const bm = seen_list + PARTS_SEEN * PARTS_BLOCK;
    PartSeen seen;
    if (r.penal) part_history(a, p, false, bm, seen_list, &s_n, seen);
    float lo0, hi0, lo1, hi1, unused;
    nuc_range(r, w0.bin, lo0, hi0);
    nuc_range(r, w1.bin, unused, hi1);
    nuc_range(r, w2.bin, lo1, unused);
    const NucList staged{stage + wave_id() * WCAP, &s_wcount[wave_id()]};
    staged.clear();
    auto wanted = [&](float y) { return nuc_within(y, lo0, hi0) | nuc_within(y, lo1, hi1); };
    auto append = [&](float y, int j) { staged.append<WCAP>(wanted(y), y, j); };
    nuc_foreach4<PARTS_BLOCK, true, true, true>(r, bm, [&](int j, const float (&y)[4]) { staged.append4<WCAP>(wanted, y, j); },
                                                [&](int j, float y) { append(y, j); }, NucNoPre(), first);
    if (r.penal) {
#pragma unroll
        for (int k = 0; k < PARTS_SEEN; k++)
            if (seen.id[k] >= 0) append(seen.y[k], (int)((u32)seen.id[k] | 0x80000000u));
    }
    lds_barrier();                                                   // (the seen ids' storage is free; s_n too)
    if (tid == 0) s_n = 0;
    lds_barrier();
    const long long part = (long long)row * pa.parts + blockIdx.y;
    ulonglong2 *const out = pa.list + part * PARTS_LIST;
    const u32 count = staged.size();
    if (count > (u32)WCAP && l == 0) s_over = 1;
    for (int e0 = 0; e0 < (int)min(count, (u32)WCAP); e0 += WAVE) {
        const int e = e0 + l;
        bool take = false;
        u64 key = 0ull, qs = 0ull;
        if (e < (int)min(count, (u32)WCAP)) {
            uint2 c = staged.at[e];
            bool stale = false;                                      // a seen id's stored logit
            if (r.penal) {
                if (c.y & 0x80000000u) c.y &= 0x7FFFFFFFu;
                else stale = (bm[c.y >> 5] >> (c.y & 31)) & 1u;
            }
            const float z = nuc_z(r, __uint_as_float(c.x));
            const float d = nuc_d(r, z);
            const int b = nuc_bin(r, d);
            const int slot = stale ? -1 : b >= w1.bin && b <= w2.bin ? (joined ? 0 : 1) : b == w0.bin ? 0 : -1;
            if (slot >= 0) {
                take = true;
                key = make_key64(z, p.lo + (int)c.y);
                qs = qfix(expneg(d, r.dcut), r.scale) | ((u64)slot << 62);
            }
        }
        const u64 mk = __ballot(take);
        if (mk) {
            int base = 0;
            if (l == 0) base = atomicAdd(&s_n, __popcll(mk));
            base = __builtin_amdgcn_readfirstlane(base);
            const int pos = base + (int)__builtin_amdgcn_mbcnt_hi((u32)(mk >> 32), __builtin_amdgcn_mbcnt_lo((u32)mk, 0u));
            if (take && pos < PARTS_LIST) out[pos] = make_ulonglong2(key, qs);
        }
    }
    if (tells) {
        PartsRow &to = pa.rows[row];
        to.tp = tp;
        to.Zk = Zk;
        to.before[0] = joined ? w1.before : w0.before;
        to.before[1] = w1.before;
        to.m = r.m;
        to.draw = joined ? 0 : 1;
        to.alone = 0;
    }
    lds_barrier();
    if (tid == 0) pa.count[part] = s_over ? (u32)PARTS_LIST + 1u : (u32)s_n;
}

// One workgroup per row: the parts' lists in rank order, the cut and the draw.  False: the row is the one-workgroup body's.
__device__ __forceinline__ bool nucleus_parts_draw(const SampleArgs &a, const PartsArgs &pa, float u) {
    extern __shared__ __align__(16) u64 nuc_dyn[];                   // [PARTS_CAP] keys by bucket, then keys and masses in rank order
    __shared__ BlockScratch scr;
    __shared__ u64 s_win[2], s_mass[2], s_slot0[4];
    __shared__ u32 s_start[PARTS_ROW_MAX + 1], s_top[2], s_low[2];
    __shared__ __align__(16) u32 s_count[256], s_at[256];
    __shared__ int s_over;
    const int tid = threadIdx.x, row = blockIdx.x, l = lane_id();
    u64 *const grouped = nuc_dyn, *const skey = grouped + PARTS_CAP, *const sq = skey + PARTS_CAP;
    const PartsRow &of = pa.rows[row];
    const bool alone = of.alone != 0, cut = a.top_p < 1.0f;
    const u64 tp = of.tp, Zk = of.Zk, before[2] = {of.before[0], of.before[1]};
    const int draw = of.draw;
    const float m = of.m;
    if (tid < 2) s_win[tid] = 0ull;
    if (tid < 256) s_count[tid] = 0u;
    if (tid < 2) {
        s_top[tid] = 0u;
        s_low[tid] = ~0u;
    }
    if (tid < WAVE) {
        const u32 c = l < pa.parts ? pa.count[(long long)row * pa.parts + l] : 0u;
        const u32 upto = wave_inclusive_scan_u32(min(c, (u32)PARTS_CAP + 1u));
        if (l < pa.parts) s_start[l + 1] = upto;
        const u64 over = __ballot(c > (u32)PARTS_LIST);
        if (l == 0) {
            s_start[0] = 0u;
            s_over = over != 0ull;
        }
    }
    __syncthreads();
    if (alone) return false;                                         // (its counts are from an earlier call)
    const int n = (int)s_start[pa.parts];
    if (s_over || n > PARTS_CAP) return false;                       // workgroup-uniform
    // Every thread one entry: the part its place falls into.  Ranks through buckets, 128 for the range of either slot (the draw's bins lie
    // above the cut's): an entry counts the keys above its own in its bucket only.  (Against all others,
    // two 128-bit reads for four keys, the launch took 19 us on 32 rows of 152 064; 32 x 152 064 in all 40.9 us, 36.0 so, 64 rows 49.2 and 44.8.)
    u64 key = 0ull, qs = 0ull;
    if (tid < n) {
        int q = 0;
        for (int half = PARTS_ROW_MAX / 2; half; half >>= 1)
            if (q + half < pa.parts && s_start[q + half] <= (u32)tid) q += half;
        const ulonglong2 e = pa.list[((long long)row * pa.parts + q) * PARTS_LIST + (tid - (int)s_start[q])];
        key = e.x;
        qs = e.y;
    }
    const u32 z = (u32)(key >> 32);
    const int in_slot = (int)(qs >> 62);
    if ((tid & ~(WAVE - 1)) < n) {                                   // wave-uniform
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const bool its = tid < n && in_slot == t;
            const u32 most = wave_max_u32(its ? z : 0u), least = wave_min_u32(its ? z : ~0u);
            if (l == 0) {
                atomicMax(&s_top[t], most);
                atomicMin(&s_low[t], least);
            }
        }
    }
    lds_barrier();
    u32 bucket = 0u, pos = 0u;
    if (tid < n) {
        const u32 range = s_top[in_slot] - s_low[in_slot];
        const int sh = max(0, 25 - (int)__clz(range));               // (range >> sh) < 128
        bucket = (in_slot ? 0u : 128u) + ((s_top[in_slot] - z) >> sh);
        pos = atomicAdd(&s_count[bucket], 1u);
    }
    lds_barrier();
    if (tid < WAVE) {
        const uint4 c = reinterpret_cast<const uint4 *>(s_count)[tid];
        const u32 four = c.x + c.y + c.z + c.w, ex = wave_inclusive_scan_u32(four) - four;
        reinterpret_cast<uint4 *>(s_at)[tid] = make_uint4(ex, ex + c.x, ex + c.x + c.y, ex + c.x + c.y + c.z);
    }
    lds_barrier();
    u32 start = 0u;
    if (tid < n) {
        start = s_at[bucket];
        grouped[start + pos] = key;
    }
    lds_barrier();
    if (tid < n) {
        const u32 c = s_count[bucket];
        u32 rank = start;
        for (u32 j = 0; j < c; j++) rank += grouped[start + j] > key ? 1u : 0u;
        skey[rank] = key;
        sq[rank] = qs;
    }
    __syncthreads();
    u64 mykey = 0ull, mine = 0ull, q = 0ull, all;
    int myslot = -1;
    if (tid < n) {
        mykey = skey[tid];
        myslot = (int)(sq[tid] >> 62);
        q = sq[tid] & 0x3FFFFFFFFFFFFFFFull;
    }
    const u64 incl = block_inclusive_scan_u64<PARTS_BLOCK>(q, &scr, &all);
    if (tid < n && (tid == 0 || (int)(sq[tid - 1] >> 62) != myslot)) s_slot0[myslot] = incl - q;
    __syncthreads();
    if (tid < n) mine = incl - s_slot0[myslot];                      // the mass at and above this entry in its bin

    // ---- the cut, then the draw: the first entry in rank order at which the cumulative mass reaches the target, which its own mass crosses
    u64 Zp = Zk, tokkey = 0ull;
    for (int phase = cut ? 0 : 1; phase < 2; phase++) {
        const u64 target = phase == 0 ? tp : draw_target(u, Zp);
        const int slot = phase == 0 ? 0 : draw;
        const u64 base = slot ? before[1] : before[0];
        if (myslot == slot && base + mine >= target && base + (mine - q) < target) {
            s_win[phase] = mykey;
            s_mass[phase] = base + mine;
        }
        __syncthreads();
        const u64 win = s_win[phase];
        if (phase == 0) Zp = s_mass[0];
        else tokkey = win;
        if (win == 0ull) break;                                      // inconsistent masses: cannot happen
    }
    if (tid == 0) {
        if (tokkey == 0ull) {
            atomicOr(a.status, 4);
            a.tokens[row] = 0;
            if (a.probs) a.probs[row] = 0.0f;
        } else {
            a.tokens[row] = key64_id(tokkey);
            if (a.probs) a.probs[row] = prob_of(emass(key64_z(tokkey), m, a.dcut), Zp, a.mass_shift);
        }
        if (a.nuc_len) a.nuc_len[row] = -1;
        count_row(a.counters, row, 2);
    }
    return true;
}

__global__ __launch_bounds__(PARTS_BLOCK, 4) void nucleus_parts_draw_kernel(SampleArgs a, PartsArgs pa) {
    const float u = a.uniforms ? a.uniforms[blockIdx.x] : uniform_of(a.seed, a.step, (u64)blockIdx.x);
    if (nucleus_parts_draw(a, pa, u)) return;
    __syncthreads();
    nucleus_row_body<PARTS_BLOCK, false, true, true>(a, a.T, a.top_p, a.rep, a.dcut, 0.0f, 0.0f, nuc_reciprocal(a.T));
}

static size_t parts_max_lds(int len) { return sizeof(u32) * (size_t)(PARTS_SEEN * PARTS_BLOCK + (len + 31) / 32); }
static size_t parts_masses_lds(int len) { return sizeof(u64) * (NUC_BINS + NUC_BEYOND) + parts_max_lds(len); }
static size_t parts_gather_lds(int len) { return sizeof(u64) * NucGeom<PARTS_BLOCK>::WAVES * NucGeom<PARTS_BLOCK>::WCAP + parts_max_lds(len); }

static size_t parts_bytes(size_t parts) {
    return parts * (sizeof(u64) * (NUC_BINS + PARTS_RUNS) + sizeof(ulonglong2) * PARTS_LIST + sizeof(float2) + sizeof(u32) + sizeof(PartsRow));
}
static PartsArgs parts_layout(const NucleusWorkspace &ws) {
    PartsArgs pa;
    char *p = static_cast<char *>(ws.p);
    const size_t parts = (size_t)ws.parts;                           // (even: everything 16-byte aligned)
    auto take = [&p](size_t bytes) {
        char *at = p;
        p += bytes;
        return at;
    };
    pa.bins = reinterpret_cast<u64 *>(take(sizeof(u64) * NUC_BINS * parts));
    pa.runs = reinterpret_cast<u64 *>(take(sizeof(u64) * PARTS_RUNS * parts));
    pa.list = reinterpret_cast<ulonglong2 *>(take(sizeof(ulonglong2) * PARTS_LIST * parts));
    pa.ends = reinterpret_cast<float2 *>(take(sizeof(float2) * parts));
    pa.count = reinterpret_cast<u32 *>(take(sizeof(u32) * parts));
    pa.rows = reinterpret_cast<PartsRow *>(take(sizeof(PartsRow) * parts));
    pa.parts = pa.len = 0;
    return pa;
}
int nucleus_workspace_parts(int64_t max_batch) { return (int)std::min<int64_t>(PARTS_TOTAL, max_batch * PARTS_ROW_MAX); }
size_t nucleus_workspace_bytes(int parts) { return parts_bytes((size_t)parts); }
// Whether a batch's rows are cut into parts, and into how many (below 2: not).
static int parts_of(const SampleArgs &a, bool two_per_cu, int most) {
    if (two_per_cu || a.hist_counts || a.hist_stride > PARTS_SEEN * PARTS_BLOCK) return 0;
    if (a.dcut != 80.0f) return 0;                                   // (a min-p bound is for the one-workgroup body)
    return row_parts(a.V, a.B, std::min(most, device_cu_count()));
}
bool nucleus_wants_parts(const SampleArgs &a, bool two_per_cu) { return parts_of(a, two_per_cu, PARTS_TOTAL) >= 2; }
static bool parts_plan(const SampleArgs &a, bool two_per_cu, const NucleusWorkspace &ws, PartsArgs &pa) {
    const int parts = ws.p ? parts_of(a, two_per_cu, ws.parts) : 0;
    if (parts < 2) return false;
    const int len = ((a.V + parts - 1) / parts + 31) & ~31;
    pa = parts_layout(ws);
    pa.len = len;
    pa.parts = (a.V + len - 1) / len;
    return true;
}

static hipError_t launch_parts(const SampleArgs &a, const PartsArgs &pa, hipStream_t st) {
    const dim3 gr((unsigned)a.B, (unsigned)pa.parts), bl(PARTS_BLOCK);
    hipLaunchKernelGGL(nucleus_parts_max_kernel, gr, bl, parts_max_lds(pa.len), st, a, pa);
    hipLaunchKernelGGL(nucleus_parts_masses_kernel, gr, bl, parts_masses_lds(pa.len), st, a, pa);
    hipLaunchKernelGGL(nucleus_parts_gather_kernel, gr, bl, parts_gather_lds(pa.len), st, a, pa);
    hipLaunchKernelGGL(nucleus_parts_draw_kernel, dim3((unsigned)a.B), bl, nucleus_lds_bytes(a.V), st, a, pa);
    return hipGetLastError();
}

static hipError_t configure_parts() {
    const int most = (int)WIDE_MAX_VOCAB / 2 + 32;                   // (logits of a part)
    const struct {
        const void *kernel;
        size_t lds;
    } all[] = {{reinterpret_cast<const void *>(nucleus_parts_max_kernel), parts_max_lds(most)},
               {reinterpret_cast<const void *>(nucleus_parts_masses_kernel), parts_masses_lds(most)},
               {reinterpret_cast<const void *>(nucleus_parts_gather_kernel), parts_gather_lds(most)},
               {reinterpret_cast<const void *>(nucleus_parts_draw_kernel), nucleus_lds_bytes((int)WIDE_MAX_VOCAB)}};
    for (const auto &k : all) {
        const hipError_t e = hipFuncSetAttribute(k.kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)k.lds);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace born
