// Speculative-decoding accept / reject with residual max(0, p - q) resampling
// (docs/SAMPLING_SPEC.md section 5, fixed-point layer).  Three launches:
//
//   spec_stats_kernel     one workgroup per (sequence, position, distribution): row maximum and integer
//                         normaliser of the target or the draft distribution, and its mass of the draft token.
//                         Vocabularies of at most 32768 are held in registers, so each logit is read
//                         from HBM once; larger ones are swept twice.
//   spec_residual_kernel  SPEC_CHUNKS workgroups per sequence: first rejected position (every workgroup
//                         of a sequence derives it from the statistics), then the integer mass of
//                         max(0, p - q) over the workgroup's quarter of that one row.
//   spec_pick_kernel      one workgroup per sequence: the per-thread masses of the quarter the residual
//                         draw falls into are scanned and the owning thread walks its ids in ascending order.
// 64 sequences of 5 + 1 positions, 32 000 logits, us by launch: 24.2 + 12.4 + 6.5 before, 22.3 + 7.7 + 4.3 with the masses summed in fp64 (mass_sum_add), runs
// read by 128-bit loads and picked from by a wave; 42.2 -> 33.5 a step.  The statistics are bound by the vector arithmetic of their masses
// and the rows' read (92 MB), one after the other in each workgroup, at 2.75 rows a CU.  128 256 logits, 32 sequences, two sweeps with four loads in flight: 142 -> 86.
// With bonus rows (the target's distribution one position past the draft) a sequence without a rejection draws
// its next token from that row the same way: the "residual" is then the row's own integer masses.
#include "dev_common.h"
#include "kernels.h"

namespace born {

constexpr int SPEC_BLOCK = 1024;
constexpr int SPEC_NF4 = 8;                   // float4 per thread and array that the stats kernel keeps in registers
// Rows that start at any four bytes are read by 128-bit loads from this length on (600 x 3 x 1001: 48.5 us one logit at a time, 49.9 by
// 128-bit loads; 2039 55.6 and 53.1; 3001 62.6 and 56.2).
constexpr int SPEC_LOADS4_FROM = 1536;
constexpr int SPEC_RESIDENT_V = SPEC_NF4 * SPEC_BLOCK * 4;

typedef row_f32x4 spec_f32x4;

// The logits of a row in blocks of four, SPEC_FLIGHT loads of a thread in flight together, then its last V % 4: f4(block), f1(logit).
constexpr int SPEC_FLIGHT = 4;
template <class F4, class F1>
__device__ __forceinline__ void spec_blocks(const float *x, int V, F4 f4, F1 f1) {
    const int tid = threadIdx.x, n4 = V >> 2;
    const spec_f32x4 *x4 = reinterpret_cast<const spec_f32x4 *>(x);
    int i = tid;
    for (; i + (SPEC_FLIGHT - 1) * SPEC_BLOCK < n4; i += SPEC_FLIGHT * SPEC_BLOCK) {
        spec_f32x4 q[SPEC_FLIGHT];
#pragma unroll
        for (int k = 0; k < SPEC_FLIGHT; k++) q[k] = x4[i + k * SPEC_BLOCK];
#pragma unroll
        for (int k = 0; k < SPEC_FLIGHT; k++) f4(q[k]);
    }
    for (; i < n4; i += SPEC_BLOCK) f4(x4[i]);
    for (int j = (n4 << 2) + tid; j < V; j += SPEC_BLOCK) f1(x[j]);
}

// One workgroup per (sequence, position, distribution): blockIdx.x = 2 * row + (0 target | 1 draft).  The two
// distributions of a position are independent, and twice as many work items spread better over the CUs.
// RESIDENT: V <= SPEC_RESIDENT_V and a row that 128-bit loads suit (SpecArgs::wide).  TAIL: V may be no multiple of four.
// z = canon(x / T); UNIT: T == 1, where the division is the identity and is not computed at all.
template <bool UNIT>
__device__ __forceinline__ float spec_z(float x, float T, float rcp) {
    if (!UNIT) return rcp != 0.0f ? z_of_shortcut(x, T, rcp) : z_of(x, T);
    // a logit of ordinary magnitude (2^-100 <= |x| < 2^100) is its own canonical form: one integer range test, and a
    // branch that waves of ordinary logits never take, instead of three compares and selects on every logit
    if (ordinary_magnitude(x)) return x;
    asm volatile("" ::: "memory");                                   // (keeps the rest behind a branch)
    return canon(x);
}

// The usual row: a maximum m = z(largest logit) of ordinary size (2^-40 <= |m| < 2^60) and, away from temperature 1, a
// temperature whose division has the three-instruction shortcut.  The integer mass of a logit x of such a row needs no
// test of x: with z' the shortcut's quotient (x itself at temperature 1), it is that of exp(clamp(z' - m, -87, 0)):
//   2^-100 <= |x| < 2^100  z' is the correctly rounded quotient, a canonical z;
//   zeros, |x| < 2^-100    z' stays below 2^-78, less than half an ulp of m: z' - m = -m, as with the exact z;
//   -inf, NaN              z' - m is -inf or a NaN; the clamp (a median of three, which returns the smallest operand
//                          when one is a NaN) gives -87: no mass, as specified for z = -inf;
//   x <= -2^100            z' is -inf or far below m - 80: no mass;
//   +inf, x >= 2^100       not in such a row.
// Beyond d = 80 the specified mass is 0, and so is trunc(exp(-d) * 2^S) down to the clamp (S <= 61).
__device__ __forceinline__ bool spec_usual_row(float m, float T, float rcp) {
    const float am = fabsf(m);
    return am >= 0x1p-40f && am < 0x1p60f && (T == 1.0f || rcp != 0.0f);
}
template <bool UNIT>
__device__ __forceinline__ float spec_usual_e(float x, float m, float T, float rcp) {
    float z = x;
    if (!UNIT) {
        const float q = __fmul_rn(x, rcp), e = __fmaf_rn(-q, T, x);
        z = __fmaf_rn(e, rcp, q);
    }
    return expneg_core(__builtin_amdgcn_fmed3f(z - m, -87.0f, 0.0f));
}
template <bool UNIT>
__device__ __forceinline__ u64 spec_usual_mass(float x, float m, float T, float rcp, float scale32) {
    return qfix32(spec_usual_e<UNIT>(x, m, T, rcp), scale32);
}

template <bool RESIDENT, bool UNIT, bool TAIL>
__global__ __launch_bounds__(SPEC_BLOCK) void spec_stats_kernel(SpecArgs a) {
    __shared__ BlockScratch scr;
    const int tid = threadIdx.x;
    const int V = a.V;
    const bool is_bonus = (int)blockIdx.x >= 2 * a.B * a.G;          // the workgroups after the (position, distribution) pairs
    const int row = is_bonus ? (int)blockIdx.x - 2 * a.B * a.G : (int)(blockIdx.x >> 1);   // bonus: the sequence
    const bool is_draft = !is_bonus && (blockIdx.x & 1);
    const float *x = is_bonus ? a.bonus + (long long)row * a.b_seq
                              : (is_draft ? a.draft + (long long)(row / a.G) * a.d_seq : a.target + (long long)(row / a.G) * a.t_seq) +
                                    (long long)(row % a.G) * V;
    const float T = a.T, rcp = a.rcp_T;
    const float scale = mass_scale(a.mass_shift);
    // The draft token and its logit are two dependent loads: requested now, used after the reductions (at the end of
    // the kernel they would be two memory round trips nothing overlaps).
    int dt = -1;
    float xdt = 0.0f;
    if (tid == 0 && !is_bonus) {
        dt = a.draft_tokens[row];
        if (dt >= 0 && dt < V) xdt = x[dt];
    }
    float m = -INFINITY;
    u64 sum = 0;
    if (RESIDENT) {
        const int n4 = V >> 2;
        spec_f32x4 t[SPEC_NF4];
        const int jt = TAIL ? (n4 << 2) + tid : V;                   // the row's last V % 4 logits, one per thread
        float last = -INFINITY;
        if (TAIL && jt < V) last = x[jt];
        m = fmaxf(m, last);
#pragma unroll
        for (int i = 0; i < SPEC_NF4; i++) {
            const int j = i * SPEC_BLOCK + tid;
            const spec_f32x4 fill = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
            t[i] = j < n4 ? __builtin_nontemporal_load(reinterpret_cast<const spec_f32x4 *>(x) + j) : fill;
        }
        // (z is a non-decreasing function of the logit: the maximum of the logits as stored, NaNs ignored, gives m)
#pragma unroll
        for (int i = 0; i < SPEC_NF4; i++) {
#pragma unroll
            for (int c = 0; c < 4; c++) m = fmaxf(m, t[i][c]);
        }
        m = block_max_f32<SPEC_BLOCK>(m, &scr);
        m = UNIT ? canon(m) : spec_z<false>(m, T, rcp);
        if (spec_usual_row(m, T, rcp)) {                             // (uniform)
            const float scale32 = scale * 2.3283064365386963e-10f;
            if (a.mass_shift <= 50) {
                // V >= 2048: a thread's logits are at most 2^(52 - S) in number (S = 62 - bitlen(V)), so their masses fit one fp64 sum;
                // a shorter row has a block a thread at most
                const double start = mass_sum_start(a.mass_shift);
                double acc = start;
                mass_sum_begin(acc);
#pragma unroll
                for (int i = 0; i < SPEC_NF4; i++) {
                    if (i * SPEC_BLOCK + tid < n4) {
#pragma unroll
                        for (int c = 0; c < 4; c++) mass_sum_add(acc, spec_usual_e<UNIT>(t[i][c], m, T, rcp));
                    }
                }
                mass_sum_end(acc);
                sum = mass_sum_of(acc, start);
            } else if (tid < n4) {
#pragma unroll
                for (int c = 0; c < 4; c++) sum += spec_usual_mass<UNIT>(t[0][c], m, T, rcp, scale32);
            }
            if (TAIL && jt < V) sum += spec_usual_mass<UNIT>(last, m, T, rcp, scale32);
        } else if (m > -INFINITY) {                                  // (uniform) m - z is a number: +inf for a masked logit, no mass
#pragma unroll
            for (int i = 0; i < SPEC_NF4; i++) {
                if (i * SPEC_BLOCK + tid < n4) {
#pragma unroll
                    for (int c = 0; c < 4; c++) sum += qfix(expneg(m - spec_z<UNIT>(t[i][c], T, rcp)), scale);
                }
            }
            if (TAIL && jt < V) sum += qfix(expneg(m - spec_z<UNIT>(last, T, rcp)), scale);
        } else {                                                     // nothing finite: (-inf) - (-inf) := 0 for every logit
#pragma unroll
            for (int i = 0; i < SPEC_NF4; i++) {
                if (i * SPEC_BLOCK + tid < n4) {
#pragma unroll
                    for (int c = 0; c < 4; c++) sum += qfix(emass(spec_z<UNIT>(t[i][c], T, rcp), m), scale);
                }
            }
            if (TAIL && jt < V) sum += qfix(emass(spec_z<UNIT>(last, T, rcp), m), scale);
        }
    } else if (a.wide) {                                             // more than SPEC_RESIDENT_V logits, read twice
        spec_blocks(x, V, [&](const spec_f32x4 &q) {
#pragma unroll
            for (int c = 0; c < 4; c++) m = fmaxf(m, q[c]);
        }, [&](float v) { m = fmaxf(m, v); });
        m = block_max_f32<SPEC_BLOCK>(m, &scr);
        m = UNIT ? canon(m) : spec_z<false>(m, T, rcp);
        if (spec_usual_row(m, T, rcp)) {                             // (uniform)
            const float scale32 = scale * 2.3283064365386963e-10f;
            const double start = mass_sum_start(a.mass_shift);       // (a thread's logits in whole blocks are at most 2^(52 - S) here too)
            double acc = start;
            mass_sum_begin(acc);
            float last = -INFINITY;                                  // (one of the row's last three: apart, the sum may be full)
            spec_blocks(x, V, [&](const spec_f32x4 &q) {
#pragma unroll
                for (int c = 0; c < 4; c++) mass_sum_add(acc, spec_usual_e<UNIT>(q[c], m, T, rcp));
            }, [&](float v) { last = v; });
            mass_sum_end(acc);
            sum = mass_sum_of(acc, start) + spec_usual_mass<UNIT>(last, m, T, rcp, scale32);
        } else {
            auto add = [&](float v) { sum += qfix(emass(spec_z<UNIT>(v, T, rcp), m), scale); };
            spec_blocks(x, V, [&](const spec_f32x4 &q) {
#pragma unroll
                for (int c = 0; c < 4; c++) add(q[c]);
            }, add);
        }
    } else {                                                         // fewer than SPEC_LOADS4_FROM, one at a time
        for (int j = tid; j < V; j += SPEC_BLOCK) m = fmaxf(m, spec_z<UNIT>(x[j], T, rcp));
        m = block_max_f32<SPEC_BLOCK>(m, &scr);
        for (int j = tid; j < V; j += SPEC_BLOCK) sum += qfix(emass(spec_z<UNIT>(x[j], T, rcp), m), scale);
    }
    u64 Z;
    block_inclusive_scan_u64<SPEC_BLOCK>(sum, &scr, &Z);
    if (tid == 0 && is_bonus) {
        a.mb[row] = m;
        a.Zb[row] = Z;
    } else if (tid == 0) {
        u64 md = 0;                                                  // mass of the draft token in this distribution
        if (dt >= 0 && dt < V) md = qfix(emass(z_of(xdt, T), m), scale);
        else atomicOr(a.status, 2);
        if (is_draft) { a.mq[row] = m; a.Zq[row] = Z; a.qd[row] = md; }
        else { a.mp[row] = m; a.Zp[row] = Z; a.pd[row] = md; }
    }
}

// ip = 1 / Zp and iq = 1 / Zq are formed once per row; each product below is one fp64 rounding.
__device__ __forceinline__ float spec_z_any(float x, float T, float rcp) {
    return rcp != 0.0f ? z_of_shortcut(x, T, rcp) : z_of(x, T);      // (uniform; z_of itself skips the division at T = 1)
}
// USUAL: both rows are usual ones (spec_usual_row): the masses without a test of the logits.
template <bool USUAL>
__device__ __forceinline__ u64 residual_mass(float t, float d, float T, float rcp, float mp, float mq, float scale, double ip,
                                             double iq, double scale_d) {
    u64 mt, md;
    if (USUAL) {
        const float scale32 = scale * 2.3283064365386963e-10f;
        if (T == 1.0f) {                                             // (uniform)
            mt = spec_usual_mass<true>(t, mp, T, rcp, scale32);
            md = spec_usual_mass<true>(d, mq, T, rcp, scale32);
        } else {
            mt = spec_usual_mass<false>(t, mp, T, rcp, scale32);
            md = spec_usual_mass<false>(d, mq, T, rcp, scale32);
        }
    } else {
        mt = qfix(emass(spec_z_any(t, T, rcp), mp), scale);
        md = qfix(emass(spec_z_any(d, T, rcp), mq), scale);
    }
    double pj = (double)mt * ip;
    double qj = (double)md * iq;
    double r = pj > qj ? pj - qj : 0.0;
    return (u64)(r * scale_d);
}

// What the statistics hold of a sequence's positions: lane i has position i's (the first 64 of them), requested together, so that the
// rejected one's is at hand as soon as it is known and not a memory round trip later.
struct SpecLanes {
    float mp, mq, mb;             // mb: of the bonus row
    u64 Zp, Zq;
};
__device__ __forceinline__ SpecLanes spec_lanes(const SpecArgs &a, int b) {
    SpecLanes s;
    const int row = b * a.G + min(lane_id(), a.G - 1);
    s.mp = a.mp[row];
    s.mq = a.mq[row];
    s.Zp = a.Zp[row];
    s.Zq = a.Zq[row];
    s.mb = a.bonus ? a.mb[b] : 0.0f;
    return s;
}
// First position of sequence b whose draft token is rejected (G if none): accept iff u * q(d) * Zp < p(d) * Zq.
// Called by whole waves: lane i tests positions i, i + 64, ...; the lowest rejecting position wins.
__device__ __forceinline__ int spec_first_rejection(const SpecArgs &a, int b, const SpecLanes &s) {
    for (int i0 = 0; i0 < a.G; i0 += WAVE) {
        const int i = i0 + lane_id();
        bool reject = false;
        if (i < a.G) {
            const int row = b * a.G + i;
            const double lhs = (double)a.u_acc[row] * (double)a.qd[row] * (double)(i0 ? a.Zp[row] : s.Zp);
            const double rhs = (double)a.pd[row] * (double)(i0 ? a.Zq[row] : s.Zq);
            reject = !(lhs < rhs);
        }
        const u64 m = __ballot(reject);
        if (m) return i0 + __builtin_ctzll(m);
    }
    return a.G;
}

// The ids of a row are cut into SPEC_CHUNKS quarters, each quarter into one contiguous run per thread, so that
// thread order is ascending id order; runs are one id long, or whole blocks of four.  Returns the run [j0, j1) of this thread in quarter c.
// (Blocks of four in a quarter that has a thread for each id: 200 sequences of 1500 28.5 -> 32 us.)
__device__ __forceinline__ void spec_run(int V, int c, int tid, int &j0, int &j1) {
    const int per_chunk = ((V + SPEC_CHUNKS - 1) / SPEC_CHUNKS + 3) & ~3;
    const int lo = min(c * per_chunk, V), hi = min(lo + per_chunk, V);
    const int per = per_chunk <= SPEC_BLOCK ? 1 : ((per_chunk + SPEC_BLOCK - 1) / SPEC_BLOCK + 3) & ~3;
    j0 = min(lo + tid * per, hi);
    j1 = min(j0 + per, hi);
}

struct SpecRow {
    const float *xt, *xd;
    float T, rcp, mp, mq, scale;
    double Zp, Zq, scale_d;       // Zp, Zq: reciprocals of the integer normalisers
    int V;
    bool plain;                   // bonus row: the mass of id j is the row's own integer mass, there is no draft
    bool usual;                   // both maxima are of ordinary size and the division has its shortcut: masses without tests
};
__device__ __forceinline__ u64 spec_lane_u64(u64 x, int l) {
    return ((u64)(u32)__builtin_amdgcn_readlane((int)(u32)(x >> 32), l) << 32) | (u32)__builtin_amdgcn_readlane((int)(u32)x, l);
}
// Position i (uniform) of sequence b; i == G is the bonus row.
__device__ __forceinline__ SpecRow spec_row(const SpecArgs &a, int b, int i, const SpecLanes &s) {
    SpecRow r;
    r.T = a.T;
    r.rcp = a.rcp_T;
    r.scale = mass_scale(a.mass_shift);
    r.scale_d = ldexp(1.0, a.mass_shift);
    r.plain = i == a.G;
    r.V = a.V;
    u64 Zp = 1, Zq = 1;
    if (r.plain) {
        r.xt = r.xd = a.bonus + (long long)b * a.b_seq;
        r.mp = r.mq = uniform_f32(s.mb);
    } else {
        const int row = b * a.G + i;
        r.xt = a.target + (long long)b * a.t_seq + (long long)i * a.V;
        r.xd = a.draft + (long long)b * a.d_seq + (long long)i * a.V;
        if (i < WAVE) {                                              // (uniform)
            r.mp = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s.mp), i));
            r.mq = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s.mq), i));
            Zp = spec_lane_u64(s.Zp, i);
            Zq = spec_lane_u64(s.Zq, i);
        } else {
            r.mp = a.mp[row];
            r.mq = a.mq[row];
            Zp = a.Zp[row];
            Zq = a.Zq[row];
        }
    }
    r.Zp = 1.0 / (double)Zp;
    r.Zq = 1.0 / (double)Zq;
    r.usual = spec_usual_row(r.mp, r.T, r.rcp) && spec_usual_row(r.mq, r.T, r.rcp);
    return r;
}
__device__ __forceinline__ u64 spec_mass(const SpecRow &r, float t, float d) {
    if (r.plain) return qfix(emass(spec_z_any(t, r.T, r.rcp), r.mp), r.scale);    // uniform per row
    if (r.usual) return residual_mass<true>(t, d, r.T, r.rcp, r.mp, r.mq, r.scale, r.Zp, r.Zq, r.scale_d);
    return residual_mass<false>(t, d, r.T, r.rcp, r.mp, r.mq, r.scale, r.Zp, r.Zq, r.scale_d);
}
constexpr int SPEC_RUN = 8;                   // ids that a thread loads before any arithmetic: the whole run up to 32 768 ids
// Ids j .. j + 7 of both rows, those from j1 on (which are not looked at) as zeros; 128-bit loads, of rows that may start at any four
// bytes.  Only the thread that holds the row's last V % 4 ids loads them one at a time.  (One id at a time the 64 lanes of a load fetch 64 pieces
// of four bytes, 32 bytes apart: at 64 sequences of 32 000 the residual launch took 12.3 us, 8.1 like this, and 7.9 with its masses in fp64.)
__device__ __forceinline__ void spec_load_run(const SpecRow &r, int j, int j1, float (&tv)[SPEC_RUN], float (&dv)[SPEC_RUN]) {
#pragma unroll
    for (int i = 0; i < SPEC_RUN; i += 4) {
        spec_f32x4 t = {0.0f, 0.0f, 0.0f, 0.0f}, d = t;
        if (j + i + 3 < j1) {
            t = *reinterpret_cast<const spec_f32x4 *>(r.xt + j + i);
            d = *reinterpret_cast<const spec_f32x4 *>(r.xd + j + i);
        } else if (j + i < j1) {
#pragma unroll
            for (int c = 0; c < 3; c++)
                if (j + i + c < j1) {
                    t[c] = r.xt[j + i + c];
                    d[c] = r.xd[j + i + c];
                }
        }
#pragma unroll
        for (int c = 0; c < 4; c++) {
            tv[i + c] = t[c];
            dv[i + c] = d[c];
        }
    }
}
__device__ __forceinline__ u64 spec_run_mass(const SpecRow &r, int j0, int j1, int mass_shift) {
    if (r.V <= SPEC_CHUNKS * SPEC_BLOCK) return j0 < j1 ? spec_mass(r, r.xt[j0], r.xd[j0]) : 0ull;   // (uniform: one id a thread)
    u64 local = 0;
    if (r.usual && !r.plain) {                                       // (uniform; S <= 49 here, where there are more than 4096 ids)
        // The integer masses as fp64 numbers scaled by 2^-S, trunc(e 2^S) 2^-S, which is what residual_mass makes of them
        // (each integer mass is below 2^53) with the scale moved into the reciprocals: the same product and difference, rounded alike.
        const double start = mass_sum_start(mass_shift);
        double ip = r.Zp * r.scale_d, iq = r.Zq * r.scale_d;
        for (int j = j0; j < j1; j += SPEC_RUN) {
            float tv[SPEC_RUN], dv[SPEC_RUN];
            spec_load_run(r, j, j1, tv, dv);
#pragma unroll
            for (int h = 0; h < SPEC_RUN; h += 4) {
                if (h && j + h >= j1) break;                         // (runs of four ids)
                double mt[4], md[4];
                asm volatile("" : "+v"(local));                      // (the four before are done)
                mass_sum_begin(ip, iq);
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    mt[i] = md[i] = start;
                    mass_sum_add(mt[i], r.T == 1.0f ? spec_usual_e<true>(tv[h + i], r.mp, r.T, r.rcp) : spec_usual_e<false>(tv[h + i], r.mp, r.T, r.rcp));
                    mass_sum_add(md[i], r.T == 1.0f ? spec_usual_e<true>(dv[h + i], r.mq, r.T, r.rcp) : spec_usual_e<false>(dv[h + i], r.mq, r.T, r.rcp));
                }
                mass_sum_end(mt, md);
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const double pj = (mt[i] - start) * ip, qj = (md[i] - start) * iq;
                    const double d = pj > qj ? pj - qj : 0.0;
                    if (j + h + i < j1) local += (u64)(d * r.scale_d);
                }
            }
        }
        return local;
    }
    for (int j = j0; j < j1; j += SPEC_RUN) {
        float tv[SPEC_RUN], dv[SPEC_RUN];
        spec_load_run(r, j, j1, tv, dv);
#pragma unroll
        for (int i = 0; i < SPEC_RUN; i++)
            if (j + i < j1) local += spec_mass(r, tv[i], dv[i]);
    }
    return local;
}

__global__ __launch_bounds__(SPEC_BLOCK) void spec_residual_kernel(SpecArgs a) {
    __shared__ BlockScratch scr;
    const int b = blockIdx.x / SPEC_CHUNKS, c = blockIdx.x % SPEC_CHUNKS, tid = threadIdx.x;
    __shared__ SpecRow s_row;
    __shared__ int s_first;
    if (tid < WAVE) {                                                // (one wave: by each for itself the launch takes 8.9 us for 8.1)
        const SpecLanes lanes = spec_lanes(a, b);
        const int first = spec_first_rejection(a, b, lanes);
        if (first < a.G || a.bonus) {
            const SpecRow r = spec_row(a, b, first, lanes);
            if (tid == 0) s_row = r;
        }
        if (tid == 0) {
            s_first = first;
            if (c == 0) {
                a.n_accepted[b] = first;
                if (first == a.G && !a.bonus) a.next_token[b] = -1;
            }
        }
    }
    __syncthreads();
    if (s_first == a.G && !a.bonus) return;
    const SpecRow r = s_row;
    int j0, j1;
    spec_run(a.V, c, tid, j0, j1);
    const u64 local = spec_run_mass(r, j0, j1, a.mass_shift);
    a.run_mass[(long long)blockIdx.x * SPEC_BLOCK + tid] = local;    // the pick reads the quarter it needs
    u64 R;
    block_inclusive_scan_u64<SPEC_BLOCK>(local, &scr, &R);
    if (tid == 0) a.part[b * SPEC_CHUNKS + c] = R;
}

__global__ __launch_bounds__(SPEC_BLOCK) void spec_pick_kernel(SpecArgs a) {
    __shared__ BlockScratch scr;
    __shared__ float s_bv[SPEC_BLOCK / WAVE];
    __shared__ int s_bi[SPEC_BLOCK / WAVE];
    const int b = blockIdx.x, tid = threadIdx.x;
    const int G = a.G, V = a.V;
    const SpecLanes lanes = spec_lanes(a, b);                        // (requested along with n_accepted, which the residual launch wrote)
    const float u_res = a.u_res[b];
    u64 part[SPEC_CHUNKS], R = 0;
#pragma unroll
    for (int c = 0; c < SPEC_CHUNKS; c++) {
        part[c] = a.part[b * SPEC_CHUNKS + c];
        R += part[c];
    }
    const int first = __builtin_amdgcn_readfirstlane(a.n_accepted[b]);
    if (first == G && !a.bonus) return;
    if (R == 0) {
        // residual vanished in fixed point: the target's argmax, lowest id on ties
        // (never a bonus row: its maximum alone has mass 2^S)
        const float *xt = a.target + (long long)b * a.t_seq + (long long)first * V;
        float bv = -INFINITY;
        int bi = 0x7FFFFFFF;
        for (int j = tid; j < V; j += SPEC_BLOCK) {
            float z = z_of(xt[j], a.T);
            if (z > bv || (z == bv && j < bi)) { bv = z; bi = j; }
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            float ov = __shfl_xor(bv, o, WAVE);
            int oi = __shfl_xor(bi, o, WAVE);
            if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
        }
        if (lane_id() == 0) { s_bv[wave_id()] = bv; s_bi[wave_id()] = bi; }
        __syncthreads();
        if (tid == 0) {
            for (int w = 1; w < SPEC_BLOCK / WAVE; w++)
                if (s_bv[w] > bv || (s_bv[w] == bv && s_bi[w] < bi)) { bv = s_bv[w]; bi = s_bi[w]; }
            a.next_token[b] = bi;
        }
        return;
    }
    const u64 td = draw_target(u_res, R);                       // 1 <= td <= R
    int c = 0;
    u64 before = 0;                                                  // residual mass of the quarters before c
#pragma unroll
    for (int i = 0; i < SPEC_CHUNKS - 1; i++) {
        if (c == i && before + part[i] < td) {
            before += part[i];
            c = i + 1;
        }
    }
    const SpecRow r = spec_row(a, b, first, lanes);
    int j0, j1;
    spec_run(V, c, tid, j0, j1);
    const u64 local = a.run_mass[((long long)b * SPEC_CHUNKS + c) * SPEC_BLOCK + tid];
    u64 Rc;
    const u64 inc = before + block_inclusive_scan_u64<SPEC_BLOCK>(local, &scr, &Rc);
    const u64 excl = inc - local;
    const u64 owner = __ballot(excl < td && td <= inc);              // exactly one thread owns the crossing
    if (owner == 0ull) return;
    // Its wave looks for the id, one lane to each (by the owner alone the masses are a chain of some seventy instructions an id).
    const int l = __builtin_ctzll(owner), k0 = __builtin_amdgcn_readlane(j0, l), k1 = __builtin_amdgcn_readlane(j1, l);
    u64 acc = spec_lane_u64(excl, l);
    int tok = k1 - 1;
    for (int k = k0; k < k1; k += WAVE) {
        const int j = k + lane_id();
        const u64 upto = acc + wave_inclusive_scan_u64(j < k1 ? spec_mass(r, r.xt[j], r.xd[j]) : 0ull);
        const u64 hit = __ballot(j < k1 && upto >= td);
        if (hit) {
            tok = k + __builtin_ctzll(hit);
            break;
        }
        acc = spec_lane_u64(upto, WAVE - 1);
    }
    if (lane_id() == 0) a.next_token[b] = tok;
}

template <bool RESIDENT, bool TAIL>
static void launch_spec_stats(const SpecArgs &a, hipStream_t st) {
    const dim3 sg((unsigned)(2 * a.B * a.G + (a.bonus ? a.B : 0))), sb(SPEC_BLOCK);
    if (a.T == 1.0f) hipLaunchKernelGGL((spec_stats_kernel<RESIDENT, true, TAIL>), sg, sb, 0, st, a);
    else hipLaunchKernelGGL((spec_stats_kernel<RESIDENT, false, TAIL>), sg, sb, 0, st, a);
}

hipError_t launch_spec_verify(const SpecArgs &args, hipStream_t st) {
    SpecArgs a = args;
    a.wide = a.V >= SPEC_LOADS4_FROM || ((a.V & 3) == 0 && rows_aligned(a.target, a.t_seq) && rows_aligned(a.draft, a.d_seq) &&
                                       (!a.bonus || rows_aligned(a.bonus, a.b_seq)));
    if (!a.wide || a.V > SPEC_RESIDENT_V) launch_spec_stats<false, false>(a, st);
    else if (a.V & 3) launch_spec_stats<true, true>(a, st);
    else launch_spec_stats<true, false>(a, st);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(spec_residual_kernel, dim3((unsigned)(a.B * SPEC_CHUNKS)), dim3(SPEC_BLOCK), 0, st, a);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(spec_pick_kernel, dim3((unsigned)a.B), dim3(SPEC_BLOCK), 0, st, a);
    return hipGetLastError();
}

}  // namespace born
