// y = x @ W^T + b for a handful of rows of x: bound by reading the weights once.
//
// A wave owns four rows of W (columns of C) and walks along K with 128-bit loads that do not stay in the caches, two stages of
// 2 x 256 values of each row in two register sets, so that one is in flight while the other is multiplied; x comes through the L1 (16 KiB for
// one row of 4096).  No LDS and no barrier: twelve waves a CU (131 registers with one row) keep 100 to 200 KiB in flight.  The fp32 tiles
// (linear.hip) have a workgroup of four waves per CU there and a barrier every 32 values of K.  Waves start at different
// places along K, since rows a large power of two apart would crowd the same memory channels.
// Few columns: the four waves of a workgroup share a group of them and each takes a quarter of K.
// Each lane adds the products of its own values in one chain of K / 64 fused multiply-adds, then the lanes are added pairwise: shorter
// sums than the tiles' (one chain of K / 4 groups of four): 2-norm against fp64 1.6e-7 at K = 4096, theirs 1.1e-6.
//
// us, the tiles (in slices of K where the columns are few) and here, 1 and 4 rows: 4096 -> 32 000 87.6 87.6 and 72.9 82.2 (7.2 TB/s with one
// row), 4096 -> 128 256 358 360 and 289 321, 1024 -> 32 000 26.8 27.5 and 21.5 26.1, 4096 -> 4096 23.0 23.7 and 12.5 15.4, 4096 -> 1000 12.3 14.1 and
// 5.6 6.4, 784 -> 512 10.4 12.1 and 5.4 5.2.  Four rows are bound by x through the L1, as many bytes as W.
#include "gemm_epilogue.h"

namespace born {

constexpr int ROWS_NR = 4;                    // columns of C per group
constexpr int ROWS_STEP = WAVE * 4;           // values of K per load

template <int MR, int KW, int EPI>
__global__ __launch_bounds__(GEMM_THREADS) void gemm_rows_kernel(GemmArgs g) {
    constexpr int WAVES = GEMM_THREADS / WAVE, U = 2, STAGE = U * ROWS_STEP, VALUES = ROWS_NR * MR;
    static_assert(KW == 1 || KW == WAVES, "a wave, or the workgroup, per group of columns");
    static_assert(VALUES <= WAVE, "one lane per result");
    const int lane = (int)(threadIdx.x & (WAVE - 1)), wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int group = KW == 1 ? (int)blockIdx.x * WAVES + wave : (int)blockIdx.x, n0 = group * ROWS_NR;
    if (KW == 1 && n0 >= g.N) return;                                // (no barrier below then)
    const int K = g.K, stages = (K + STAGE - 1) / STAGE, per = (stages + KW - 1) / KW;
    const int s0 = KW == 1 ? 0 : wave * per, count = min(per, stages - s0);   // (no stage at all: count <= 0)
    const int rot = count > 0 ? (int)((unsigned)group % (unsigned)count) : 0;

    const float *w_row[ROWS_NR], *x_row[MR];                         // uniform
#pragma unroll
    for (int r = 0; r < ROWS_NR; r++) w_row[r] = g.b + (long long)min(n0 + r, g.N - 1) * g.ldb;
#pragma unroll
    for (int m = 0; m < MR; m++) x_row[m] = g.a + (long long)min(m, g.M - 1) * g.lda;
    auto stage_of = [&](int t) {
        const int s = t + rot;
        return (s0 + (s >= count ? s - count : s)) * STAGE;
    };
    auto load = [&](int t, f32x4 (&w)[U][ROWS_NR], f32x4 (&x)[U][MR]) {
        const int k0 = stage_of(t) + lane * 4;
#pragma unroll
        for (int u = 0; u < U; u++) {
            const unsigned k = (unsigned)min(k0 + u * ROWS_STEP, K - 4);
#pragma unroll
            for (int r = 0; r < ROWS_NR; r++) w[u][r] = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(w_row[r] + k));
#pragma unroll
            for (int m = 0; m < MR; m++) x[u][m] = *reinterpret_cast<const f32x4 *>(x_row[m] + k);
        }
    };
    float acc[ROWS_NR][MR];
#pragma unroll
    for (int r = 0; r < ROWS_NR; r++)
#pragma unroll
        for (int m = 0; m < MR; m++) acc[r][m] = 0.f;
    auto multiply = [&](int t, f32x4 (&w)[U][ROWS_NR], f32x4 (&x)[U][MR]) {
        const int k0 = stage_of(t);
        if (k0 + STAGE > K) {                                        // uniform: values past the end are zero
#pragma unroll
            for (int u = 0; u < U; u++) {
                const bool in = k0 + u * ROWS_STEP + lane * 4 < K;
#pragma unroll
                for (int c = 0; c < 4; c++) {
#pragma unroll
                    for (int r = 0; r < ROWS_NR; r++) w[u][r][c] = in ? w[u][r][c] : 0.f;
#pragma unroll
                    for (int m = 0; m < MR; m++) x[u][m][c] = in ? x[u][m][c] : 0.f;
                }
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int c = 0; c < 4; c++)
#pragma unroll
                for (int r = 0; r < ROWS_NR; r++)
#pragma unroll
                    for (int m = 0; m < MR; m++) acc[r][m] = __builtin_fmaf(w[u][r][c], x[u][m][c], acc[r][m]);
    };
    if (count > 0) {
        f32x4 wa[U][ROWS_NR], xa[U][MR], wb[U][ROWS_NR], xb[U][MR];
        load(0, wa, xa);
        int t = 0;
        for (; t + 2 < count; t += 2) {
            load(t + 1, wb, xb);
            __builtin_amdgcn_sched_barrier(0);
            multiply(t, wa, xa);
            load(t + 2, wa, xa);
            __builtin_amdgcn_sched_barrier(0);
            multiply(t + 1, wb, xb);
        }
        if (t + 1 < count) {
            load(t + 1, wb, xb);
            multiply(t, wa, xa);
            multiply(t + 1, wb, xb);
        } else {
            multiply(t, wa, xa);
        }
    }
    // Added over the lanes, half of the values going each way as long as a lane has several: value i = 4 m + r of row m, column
    // n0 + r ends in the lanes i << SHIFT and up.  (Every value by itself is six exchanges each: 4 x 320 -> 50 000 27 us.)
    float v[VALUES];
#pragma unroll
    for (int i = 0; i < VALUES; i++) v[i] = acc[i % ROWS_NR][i / ROWS_NR];
    constexpr int SHIFT = VALUES == 4 ? 4 : VALUES == 8 ? 3 : 2;
    static_assert(VALUES << SHIFT == WAVE, "the lanes of a value");
#pragma unroll
    for (int o = WAVE / 2, n = VALUES; o > 0; o >>= 1) {
        n >>= 1;
        const bool up = lane & o;
        if (n) {
#pragma unroll
            for (int i = 0; i < n; i++) {
                const float keep = up ? v[i + n] : v[i], send = up ? v[i] : v[i + n];
                v[i] = keep + __shfl_xor(send, o, WAVE);
            }
        } else {
            v[0] += __shfl_xor(v[0], o, WAVE);
        }
    }
    float val = v[0];
    const int at = lane >> SHIFT;
    const bool holds = (lane & ((1 << SHIFT) - 1)) == 0;
    if (KW > 1) {
        __shared__ float part[KW][VALUES];
        if (holds) part[wave][at] = val;
        __syncthreads();
        if (wave) return;
        val = part[0][at];
#pragma unroll
        for (int w = 1; w < KW; w++) val += part[w][at];
    }
    const int row = at / ROWS_NR, col = n0 + at % ROWS_NR;
    const bool mine = holds && row < g.M && col < g.N;
    if (g.bias && mine) val = val + g.bias[col];
    if (EPI == 0) {
        if (mine) g.c[(long long)row * g.ldc + col] = val;
    } else if (EPI == 1) {
        u64 key = mine ? gemm_argmax_key(val, col) : 0ull;
#pragma unroll
        for (int o = 1 << SHIFT; o < ROWS_NR << SHIFT; o <<= 1) key = gemm_max_u64(key, gemm_shfl_xor_u64(key, o));
        if (holds && at % ROWS_NR == 0 && row < g.M && key) gemm_offer_key(g.best, row, key);
    } else {
        if (mine) gemm_offer_candidate(g, row, col, val, g.thr[row]);
    }
}

// Columns from which a wave takes a group by itself: fewer of them would leave CUs without work.
constexpr int ROWS_ALONE_FROM = 8192;

template <int MR, int EPI>
static void launch_gemm_rows_as(const GemmArgs &g, hipStream_t st) {
    const int groups = (g.N + ROWS_NR - 1) / ROWS_NR;
    const dim3 bl(GEMM_THREADS);
    if (g.N >= ROWS_ALONE_FROM || g.K <= 2 * ROWS_STEP) hipLaunchKernelGGL((gemm_rows_kernel<MR, 1, EPI>), dim3((unsigned)((groups + 3) / 4)), bl, 0, st, g);
    else hipLaunchKernelGGL((gemm_rows_kernel<MR, 4, EPI>), dim3((unsigned)groups), bl, 0, st, g);
}
template <int EPI>
static void launch_gemm_rows_epi(const GemmArgs &g, hipStream_t st) {
    if (g.M == 1) launch_gemm_rows_as<1, EPI>(g, st);
    else if (g.M == 2) launch_gemm_rows_as<2, EPI>(g, st);
    else launch_gemm_rows_as<4, EPI>(g, st);
}

// Up to four rows; eight read x as often as W and are slower (8 x 4096 -> 32 000 103 us, the tiles 88).  A wave's adding over the lanes is what
// many columns and a short K take, and lanes past a short K idle; the tiles have it where they are at their best, in one round of 256 or fewer (us, tiles
// and here):
//   one row, K a multiple of 32   K = 64, 12 000 columns 4.1 4.2, 20 000 4.1 4.9, 50 000 4.5 8.6, 152 064 9.7 27.6;   192, 20 000 5.4 5.2;
//                                 256, 50 000 9.6 11.7, 100 000 20.7 21.9;   320, 30 000 8.0 7.8, 50 000 12.8 12.2;   384, 152 064 35.7 36.1
//   other K (guarded tiles)       20, 18 000 5.2 4.6, 152 064 10.0 23.5;   100, 30 000 7.3 6.5, 50 000 8.4 9.0;   200, 100 000 22.3 21.3;   260, 152 064 33.8 32.8
//   two rows and more             320, 50 000, 2 and 4 rows 15.4 16.0 and 17.9 24.7;   1024, 10 000 12.9 7.4 and 13.3 8.4, 50 000 32.2 29.9 and 32.7 33.9
//   three and four                1024, 32 000 20.5 21.6 and 20.8 22.4;   2048, 32 000 39.9 40.4 and 40.6 43.1, 50 000 73.7 63.0 and 74.5 67.4;   4096, 32 000 87.2 78.1 and 87.3 82.4
bool gemm_rows_takes(const GemmArgs &g, bool b_transposed) {
    if (!b_transposed || g.bm || g.M > GEMM_ROWS_MAX || !g.vec_a || !g.vec_b || g.K % 4) return false;
    if (g.M == 1) {
        if (g.K % 32) return g.N < 24576 || (long long)g.K * 512 >= g.N;
        return g.N < 16384 || g.K >= (g.N < 24576 ? 192 : 320);
    }
    if (g.N < ROWS_ALONE_FROM) return true;
    return g.K >= (g.M > 2 && g.N > 24576 && g.N <= 32768 ? 3072 : 1024);
}
hipError_t launch_gemm_rows(const GemmArgs &g, hipStream_t st) {
    if (g.cand) launch_gemm_rows_epi<2>(g, st);
    else if (g.best) launch_gemm_rows_epi<1>(g, st);
    else launch_gemm_rows_epi<0>(g, st);
    return hipGetLastError();
}

}  // namespace born
