// The kernels that take rows without a top-k cut (nucleus_row_impl.h: the row's body), and the log-probability of a given token.
#include "nucleus_row_impl.h"

// (the general kernel's row body, for the kernel below that takes a row of either kind)
#define BORN_WIDE_BLOCK 1024
#define BORN_WIDE_NS wide_in_nucleus
#define BORN_WIDE_BODY_ONLY
#include "sample_wide_impl.h"
#undef BORN_WIDE_BODY_ONLY
#undef BORN_WIDE_BLOCK
#undef BORN_WIDE_NS

namespace born {

// (at most 128 registers either way: 512 threads are launched two workgroups to a CU)
// KEEP: see the body; off for a batch small enough to be re-read from the L2s, where the stage held in registers costs more than its loads
// (64 x 32 000: 16.9 us with it, 16.7 without; 100 x 300 12.1 and 11.8; but 256 x 128 256 61.7 and 63.4, 200 x 50 257 29.4 and 30.0).
template <int BLOCK, bool COUNTED, bool KEEP = true>
__global__ __launch_bounds__(BLOCK, 4) void nucleus_row_kernel(SampleArgs a) {
    nucleus_row_body<BLOCK, COUNTED, KEEP>(a, a.T, a.top_p, a.rep, a.dcut, a.freq, a.pres, a.rcp_T);
}
// The batch carries a configuration per row (row_config.h): the workgroup takes the row only if it is its own.
template <int BLOCK, bool COUNTED>
__global__ __launch_bounds__(BLOCK, 4) void nucleus_row_rows_kernel(SampleArgs a, RowConfigs rc) {
    RowValues v;
    bool invalid;
    if (!row_config_values(a, rc, (int)blockIdx.x, ROUTE_NUCLEUS, v, invalid)) return;   // workgroup-uniform, before any barrier
    if (invalid) {
        row_config_reject(a, (int)blockIdx.x);
        return;
    }
    nucleus_row_body<BLOCK, COUNTED, true, true>(a, v.T, v.top_p, v.rep, v.dcut, v.freq, v.pres, nuc_reciprocal(v.T));
}
// Per-row configurations of any kind: the rows without a top-k cut and the rows of the general kernel in one launch (a
// launch whose workgroups all find their rows to be another kernel's still costs its 7 us at 256 rows).
template <bool COUNTED>
__global__ __launch_bounds__(1024) void nucleus_or_general_rows_kernel(SampleArgs a, RowConfigs rc) {
    extern __shared__ __align__(16) u64 either_dyn[];                // (the same storage as the three-sweep body's)
    __shared__ BlockScratch wide_scr;
    __shared__ int wide_int[8];
    __shared__ u64 wide_u64[4];
    const int row = (int)blockIdx.x;
    RowValues v;
    bool invalid;
    if (row_config_values(a, rc, row, ROUTE_NUCLEUS, v, invalid)) {   // workgroup-uniform, before any barrier
        if (invalid) row_config_reject(a, row);
        else nucleus_row_body<1024, COUNTED, true, true>(a, v.T, v.top_p, v.rep, v.dcut, v.freq, v.pres, nuc_reciprocal(v.T));
        return;
    }
    if (!row_config(a, rc, row, ROUTE_GENERAL, invalid)) return;
    if (invalid) {
        row_config_reject(a, row);
        return;
    }
    wide_in_nucleus::wide_row<COUNTED>(a, row, (lds_u64 *)either_dyn, (BORN_LDS BlockScratch *)&wide_scr, (lds_int *)wide_int, (lds_u64 *)wide_u64);
}

// ---------------------------------------------------------------------------------------------------------
// Log-probability of one given token per row under the softmax of the row's penalised, temperature-scaled
// logits (no truncation): z[token] - logsumexp(z).  With temperature 1 and no history it is minus the per-row
// loss term of the reference's CrossEntropyLoss.Forward (internal/nn/cross_entropy.go:37-90).
//
// One workgroup per row, ONE sweep of the row: every thread keeps a running maximum m_t and the sum of
// exp(z - m_t) over its elements, rescaled when a group of four raises the maximum (a handful of times per
// thread); the workgroup then combines the 1024 pairs.  Exponentials are the hardware's (relative error about
// 1e-7), each group of four is summed in fp32 and accumulated in fp64, the combination is fp64 throughout: the
// result is a floating-point quantity, specified by its tolerance against the fp64 value (1e-5 + 1e-6 |value|),
// not bit for bit.
// ---------------------------------------------------------------------------------------------------------
__device__ __forceinline__ double wave_sum_f64(double v) {
#pragma unroll
    for (int o = WAVE / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, WAVE);
    return v;
}

// NUC_BLOCK: 1024 threads per row, or 512 for batches of more rows than the device has CUs (two rows to a CU at a time: a
// CU holds one 1024-thread workgroup of this kernel, and the rows beyond the first round would wait for a free CU).
template <int NUC_BLOCK>
__global__ __launch_bounds__(NUC_BLOCK, 4) void token_logprob_kernel(SampleArgs a, const int *__restrict__ tokens,
                                                                     float *__restrict__ out) {
    constexpr int NUC_WAVES = NUC_BLOCK / WAVE;
    extern __shared__ __align__(16) u64 nuc_dyn[];
    __shared__ BlockScratch scr;
    __shared__ double s_part[NUC_WAVES];
    u32 *const bm = reinterpret_cast<u32 *>(nuc_dyn);                // history bitmap, one bit per id
    const int tid = threadIdx.x, row = blockIdx.x;
    const int V = a.V;

    NucRow r;
    r.x = a.logits + (long long)row * a.row_stride;
    r.V = V;
    r.n4 = V >> 2;
    r.T = a.T;
    r.rep = a.rep;
    r.scale = 0.0f;
    r.dcut = 80.0f;
    r.range = 0.0f;
    r.sbin = 0.0f;
    r.m = 0.0f;
    r.degenerate = false;
    r.counts = a.hist_counts ? a.hist_counts + (long long)row * V : nullptr;
    r.freq = a.freq;
    r.pres = a.pres;

    const int hlen = a.history ? min((int)(a.hist_len ? a.hist_len[row] : (int)a.hist_stride), (int)a.hist_stride) : 0;
    const int *h = a.history + (long long)row * a.hist_stride;
    r.penal = (a.rep != 1.0f || r.counts) && hlen > 0;
    // The queried token and its logit are two dependent loads: requested now, used after the sweep (at the end of the
    // kernel they would be two memory round trips nothing overlaps).
    int qt = -1;
    float qy = 0.0f;
    if (tid == 0) {
        qt = tokens[row];
        if (qt >= 0 && qt < V) qy = r.x[qt];
    }
    // The history bitmap is built with the row's first loads already in flight: this thread's first history entry is
    // requested before them (loads return in order), and the barriers wait for LDS traffic only.
    const int h0 = tid < hlen ? h[tid] : -1;
    auto build_bitmap = [&]() {
        if (r.penal) {
            for (int i = tid; i < ((V + 31) >> 5); i += NUC_BLOCK) bm[i] = 0u;
            lds_barrier();
        }
        for (int i = tid; i < hlen; i += NUC_BLOCK) {
            const int t = i == tid ? h0 : h[i];
            if (t < 0 || t >= V) atomicOr(a.status, 1);
            else if (r.penal) atomicOr(&bm[t >> 5], 1u << (t & 31));
        }
        lds_barrier();
    };

    // z = y / T by a reciprocal and one correction step (quotient, exact remainder, update): the correctly rounded
    // quotient but for rare last-bit cases, at a quarter of the instructions of the IEEE division the sampling
    // kernels need for their bit-exact ranks; this kernel's result is held to a tolerance.  Infinite y bypass it.
    const float rT = 1.0f / r.T;
    const bool unit = r.T == 1.0f;
    auto zof = [&](float y) {
        if (unit) return canon(y);
        const float q0 = y * rT;
        const float q1 = fmaf(fmaf(-q0, r.T, y), rT, q0);
        return canon(fabsf(y) <= 3.402823466e+38f ? q1 : q0);
    };
    // exp(z - m) with the conventions of the pipeline: a tie with the maximum is exactly 1 (also when both are -inf)
    auto term = [](float z, float m) { return z == m ? 1.0f : __expf(z - m); };
    float mt = -INFINITY;                                            // running maximum of this thread's z
    double st = 0.0;                                                 // sum of exp(z - mt) over this thread's elements
    auto raise = [&](float mnew) {                                   // mnew > mt
        st *= (double)__expf(mt - mnew);                             // exp(-inf) = 0: nothing finite was seen so far
        mt = mnew;
    };
    auto four = [&](int, const float (&y)[4]) {
        float z[4];
#pragma unroll
        for (int t = 0; t < 4; t++) z[t] = zof(y[t]);
        const float m4 = fmaxf(fmaxf(z[0], z[1]), fmaxf(z[2], z[3]));
        if (m4 > mt) raise(m4);
        st += (double)((term(z[0], mt) + term(z[1], mt)) + (term(z[2], mt) + term(z[3], mt)));
    };
    auto one = [&](int, float y) {
        const float z = zof(y);
        if (z > mt) raise(z);
        st += (double)term(z, mt);
    };
    if (r.penal) nuc_foreach4<NUC_BLOCK, true, false, false, false>(r, bm, four, one, build_bitmap);
    else nuc_foreach4<NUC_BLOCK, true, false, true, false>(r, bm, four, one, build_bitmap);

    const float m = block_max_f32<NUC_BLOCK>(mt, &scr);
    double part = mt == m ? st : st * exp((double)mt - (double)m);   // a thread without elements: st = 0
    part = wave_sum_f64(part);
    if (lane_id() == 0) s_part[wave_id()] = part;
    __syncthreads();

    if (tid == 0) {
        double S = 0.0;
#pragma unroll
        for (int w = 0; w < NUC_WAVES; w++) S += s_part[w];
        const int t = qt;
        if (t < 0 || t >= V) {
            atomicOr(a.status, 1);
            out[row] = __uint_as_float(0x7FC00000u);                 // not a token of this vocabulary
        } else {
            float y = qy;
            if (r.penal && ((bm[t >> 5] >> (t & 31)) & 1u)) y = penalise_seen(y, r.rep, r.counts, t, r.freq, r.pres);
            const float z = zof(y);
            const double d = z == m ? 0.0 : (double)m - (double)z;   // >= 0, +inf for a masked token
            out[row] = (float)(-d - log(S));
        }
    }
}

// Short rows without a history (the cross-entropy term of a classifier: ten classes, a few thousand at most): a group
// of G lanes per row, 64 / G rows to a wave, no LDS and no barrier; the same arithmetic per lane as above, the lanes of
// a group combined by butterflies.  A workgroup of 1024 threads for a row of ten logits spends its time in launches:
// 65 536 x 10 took 252 us.
template <int G>
__global__ __launch_bounds__(256) void token_logprob_small_kernel(SampleArgs a, const int *__restrict__ tokens, float *__restrict__ out) {
    const int V = a.V;
    const int gl = (int)threadIdx.x & (G - 1);                       // lane within the row's group
    const long long row = ((long long)blockIdx.x * 256 + threadIdx.x) / G;
    const bool live = row < (long long)a.B;
    const float *x = a.logits + (live ? row : 0ll) * a.row_stride;
    const float T = a.T, rT = 1.0f / T;
    const bool unit = T == 1.0f;
    auto zof = [&](float y) {
        if (unit) return canon(y);
        const float q0 = y * rT;
        const float q1 = fmaf(fmaf(-q0, T, y), rT, q0);
        return canon(fabsf(y) <= 3.402823466e+38f ? q1 : q0);
    };
    auto term = [](float z, float m) { return z == m ? 1.0f : __expf(z - m); };
    int qt = -1;
    float qy = 0.0f;
    if (live && gl == 0) {
        qt = tokens[row];
        if (qt >= 0 && qt < V) qy = x[qt];
    }
    float mt = -INFINITY;
    double st = 0.0;
    auto one = [&](float y) {
        const float z = zof(y);
        if (z > mt) {
            st *= (double)__expf(mt - z);
            mt = z;
        }
        st += (double)term(z, mt);
    };
    if (live) {
        int done = 0;
        if (G == 64) {
            const int n4 = V >> 2;
            const nuc_f32x4 *x4 = reinterpret_cast<const nuc_f32x4 *>(x);
            for (int i = gl; i < n4; i += G) {
                const nuc_f32x4 q = __builtin_nontemporal_load(x4 + i);
                float z[4];
#pragma unroll
                for (int t = 0; t < 4; t++) z[t] = zof(q[t]);
                const float m4 = fmaxf(fmaxf(z[0], z[1]), fmaxf(z[2], z[3]));
                if (m4 > mt) {
                    st *= (double)__expf(mt - m4);
                    mt = m4;
                }
                st += (double)((term(z[0], mt) + term(z[1], mt)) + (term(z[2], mt) + term(z[3], mt)));
            }
            done = n4 << 2;
        }
        for (int j = done + gl; j < V; j += G) one(x[j]);
    }
    // the group's maximum, then the sums brought to it (a lane without elements: st = 0)
    float m = mt;
#pragma unroll
    for (int o = G / 2; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, WAVE));
    double part = mt == m ? st : st * exp((double)mt - (double)m);
#pragma unroll
    for (int o = G / 2; o > 0; o >>= 1) part += __shfl_xor(part, o, WAVE);
    if (live && gl == 0) {
        if (qt < 0 || qt >= V) {
            atomicOr(a.status, 1);
            out[row] = __uint_as_float(0x7FC00000u);                 // not a token of this vocabulary
        } else {
            const float z = zof(qy);
            const double d = z == m ? 0.0 : (double)m - (double)z;
            out[row] = (float)(-d - log(part));
        }
    }
}

size_t token_logprob_lds_bytes(int V) { return sizeof(u32) * (size_t)((V + 31) / 32) + 16; }

hipError_t launch_token_logprobs(const SampleArgs &a, const int *tokens, float *out, hipStream_t st, bool two_per_cu) {
    if (!a.history && a.V <= 4096) {                                 // short rows, nothing to penalise: lanes per row by length
        const long long rows = a.B;
        if (a.V <= 16) hipLaunchKernelGGL(token_logprob_small_kernel<4>, dim3((unsigned)((rows * 4 + 255) / 256)), dim3(256), 0, st, a, tokens, out);
        else if (a.V <= 128) hipLaunchKernelGGL(token_logprob_small_kernel<16>, dim3((unsigned)((rows * 16 + 255) / 256)), dim3(256), 0, st, a, tokens, out);
        else hipLaunchKernelGGL(token_logprob_small_kernel<64>, dim3((unsigned)((rows * 64 + 255) / 256)), dim3(256), 0, st, a, tokens, out);
        return hipGetLastError();
    }
    if (two_per_cu || a.B > device_cu_count())
        hipLaunchKernelGGL(token_logprob_kernel<512>, dim3((unsigned)a.B), dim3(512), token_logprob_lds_bytes(a.V), st, a, tokens, out);
    else
        hipLaunchKernelGGL(token_logprob_kernel<1024>, dim3((unsigned)a.B), dim3(1024), token_logprob_lds_bytes(a.V), st, a, tokens, out);
    return hipGetLastError();
}

template <int BLOCK>
static size_t nucleus_lds_bytes_of(int V) {
    typedef NucGeom<BLOCK> G;
    return sizeof(u64) * (NUC_BINS + G::WAVES * G::WCAP + 2 * G::CAP) + sizeof(u32) * (size_t)((V + 31) / 32);
}
size_t nucleus_lds_bytes(int V) { return nucleus_lds_bytes_of<1024>(V); }

constexpr size_t LDS_PER_CU = 160 * 1024;

// CUs of the current device (asked once per device)
int device_cu_count() {
    static int known[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (known[dev] == 0) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        known[dev] = n;
    }
    return known[dev];
}

// A batch of at most this many bytes of logits is re-read from the L2s by sweeps 2 and 3 (eight L2s of 4 MiB).
constexpr long long NUC_L2_RESIDENT_BYTES = 16ll << 20;
template <int BLOCK>
static void launch_nucleus_of(const SampleArgs &args, hipStream_t st, const RowConfigs *rows) {
    SampleArgs a = args;
    a.row_blocks = row_blocks(args);
    const dim3 gr((unsigned)a.B), bl(BLOCK);
    const size_t lds = nucleus_lds_bytes_of<BLOCK>(a.V);
    if (rows) {
        if (a.hist_counts) hipLaunchKernelGGL((nucleus_row_rows_kernel<BLOCK, true>), gr, bl, lds, st, a, *rows);
        else hipLaunchKernelGGL((nucleus_row_rows_kernel<BLOCK, false>), gr, bl, lds, st, a, *rows);
    } else if (BLOCK == 1024 && (long long)a.B * a.V * (long long)sizeof(float) <= NUC_L2_RESIDENT_BYTES) {
        if (a.hist_counts) hipLaunchKernelGGL((nucleus_row_kernel<BLOCK, true, false>), gr, bl, lds, st, a);
        else hipLaunchKernelGGL((nucleus_row_kernel<BLOCK, false, false>), gr, bl, lds, st, a);
    } else {
        if (a.hist_counts) hipLaunchKernelGGL((nucleus_row_kernel<BLOCK, true>), gr, bl, lds, st, a);
        else hipLaunchKernelGGL((nucleus_row_kernel<BLOCK, false>), gr, bl, lds, st, a);
    }
}

}  // namespace born
#include "nucleus_parts.h"
namespace born {

// Whether launch_nucleus_row would give this batch 512 threads per row.
static bool nucleus_two_per_cu(const SampleArgs &a, bool two_per_cu) {
    return (two_per_cu || a.B > device_cu_count()) && 2 * nucleus_lds_bytes_of<512>(a.V) <= LDS_PER_CU;
}
// The rows without a top-k cut and the general kernel's rows of a batch with per-row configurations: one launch where
// the former would get a workgroup of 1024 threads anyway, else the two kernels one after the other.
hipError_t launch_nucleus_and_general_rows(const SampleArgs &args, hipStream_t st, const RowConfigs &rows, bool two_per_cu) {
    SampleArgs a = args;
    a.row_blocks = row_blocks(args);
    if (nucleus_two_per_cu(a, two_per_cu)) {
        const hipError_t e = launch_nucleus_row(a, st, &rows, two_per_cu);
        if (e != hipSuccess) return e;
        return launch_sample_wide(a, st, &rows);
    }
    const size_t lds = std::max(nucleus_lds_bytes_of<1024>(a.V), wide_lds_bytes(a.V));
    if (a.hist_counts) hipLaunchKernelGGL(nucleus_or_general_rows_kernel<true>, dim3((unsigned)a.B), dim3(1024), lds, st, a, rows);
    else hipLaunchKernelGGL(nucleus_or_general_rows_kernel<false>, dim3((unsigned)a.B), dim3(1024), lds, st, a, rows);
    return hipGetLastError();
}

hipError_t launch_nucleus_row(const SampleArgs &a, hipStream_t st, const RowConfigs *rows, bool two_per_cu, const NucleusWorkspace &ws) {
    PartsArgs pa;
    if (!rows && parts_plan(a, two_per_cu, ws, pa)) {
        SampleArgs whole = a;
        whole.row_blocks = row_blocks(a);
        return launch_parts(whole, pa, st);
    }
    // More rows than CUs, and two rows' LDS fit one CU: 512 threads per row, two rows to a CU at a time.
#ifdef BORN_NUC_FORCE_1024
    if (false) launch_nucleus_of<512>(a, st, rows);                  // (measurement builds only)
#else
    if ((two_per_cu || a.B > device_cu_count()) && 2 * nucleus_lds_bytes_of<512>(a.V) <= LDS_PER_CU) launch_nucleus_of<512>(a, st, rows);
#endif
    else launch_nucleus_of<1024>(a, st, rows);
    return hipGetLastError();
}

hipError_t configure_nucleus() {
    const int lds = (int)nucleus_lds_bytes((int)WIDE_MAX_VOCAB);
    const void *kernels[] = {reinterpret_cast<const void *>(nucleus_row_kernel<1024, false>), reinterpret_cast<const void *>(nucleus_row_kernel<1024, true>),
                             reinterpret_cast<const void *>(nucleus_row_kernel<1024, false, false>),
                             reinterpret_cast<const void *>(nucleus_row_kernel<1024, true, false>),
                             reinterpret_cast<const void *>(nucleus_row_rows_kernel<1024, false>),
                             reinterpret_cast<const void *>(nucleus_row_rows_kernel<1024, true>)};
    for (const void *k : kernels) {
        const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) return e;
    }
    const int lds512 = (int)(LDS_PER_CU / 2);
    const void *half[] = {reinterpret_cast<const void *>(nucleus_row_kernel<512, false>), reinterpret_cast<const void *>(nucleus_row_kernel<512, true>),
                          reinterpret_cast<const void *>(nucleus_row_rows_kernel<512, false>),
                          reinterpret_cast<const void *>(nucleus_row_rows_kernel<512, true>)};
    for (const void *k : half) {
        const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, lds512);
        if (e != hipSuccess) return e;
    }
    const int lds_both = (int)std::max(nucleus_lds_bytes((int)WIDE_MAX_VOCAB), wide_lds_bytes((int)WIDE_MAX_VOCAB));
    const void *both[] = {reinterpret_cast<const void *>(nucleus_or_general_rows_kernel<false>),
                          reinterpret_cast<const void *>(nucleus_or_general_rows_kernel<true>)};
    for (const void *k : both) {
        const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, lds_both);
        if (e != hipSuccess) return e;
    }
    hipError_t e = configure_parts();
    if (e != hipSuccess) return e;
    e = hipFuncSetAttribute(reinterpret_cast<const void *>(token_logprob_kernel<512>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                             (int)token_logprob_lds_bytes((int)WIDE_MAX_VOCAB));
    if (e != hipSuccess) return e;
    return hipFuncSetAttribute(reinterpret_cast<const void *>(token_logprob_kernel<1024>), hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)token_logprob_lds_bytes((int)WIDE_MAX_VOCAB));
}

}  // namespace born
