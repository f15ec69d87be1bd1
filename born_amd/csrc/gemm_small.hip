// Small products, C[M,N] = A[M,K] * B (+ bias): the layers of a classifier, bound by latency.
//
// A workgroup computes a square of 16 or 32 rows and columns (v_mfma_f32_16x16x4_f32), its waves share K: chunk c of K
// is wave c % NW's, and the waves' sums are added in order through LDS at the end.  Operands go from memory straight into
// the matrix instructions' registers, a chunk ahead: no staging, no barrier before the end, one launch; rows may start at any four
// bytes, and only the last chunk of K asks where K ends.  The tiles (linear.hip) have 16 to 128 rows of 128 columns, slices of K in a launch of
// their own that another one adds, and loads of one value where K or a pitch is odd.
//
// An accumulator is one chain of fp32 additions.  The tiles have up to sixteen slices' of it, K / 128 and 512 / tiles at most, so a wave has four here, for k modulo four:
// sixteen chains or more wherever the tiles have more than four, in the squares of 32 one a wave where they have not (their registers: 1000 x 3 -> 4001 15.6 us, 20.3 with four).
// 2-norm against fp64, tiles and here (one accumulator a wave in brackets): 64 x 784 -> 512 2.3e-7 1.2e-7 (2.0e-7), 64 x 2048 -> 1024 2.2e-7 1.6e-7 (2.9e-7),
// 497 x 1568 -> 232 2.3e-7 1.9e-7 (3.6e-7), 94 x 3211 x 101 2.8e-7 2.0e-7 (3.7e-7), 2000 x 2000 -> 100 2.9e-7 2.1e-7 (4.1e-7), 3 x 100 003 -> 252 1.5e-6 1.0e-6 (1.9e-6); the times are the same.
//
// us, tiles and here: linear 64 x 784 -> 512 12.1 5.2, 64 x 512 -> 128 8.0 4.5, 64 x 128 -> 10 4.3 3.6 (a launch after another: 3.4), 1000 x 784 -> 512 29.3 16.9,
// 179 x 686 -> 226 15.4 5.2; matmul 64 x 1024 x 128 9.5 5.8, 64 x 128 x 10 8.9 3.6, 94 x 3211 x 101 20.0 12.0.  Bound by the loads' latency and, from
// about 200 million products on, by the L2s: a square of 32 rows reads 8 bytes for 64 products.
#include "gemm_epilogue.h"
#include "gemm_plan.h"

namespace born {

// T: 16-row blocks of the square's side.  U: 128-bit loads of an operand's row per lane and chunk.  NW: waves.  ACC: accumulators of a wave, one or four.
template <bool BT, int T, int U, int NW, int ACC, int EPI>
__global__ __launch_bounds__(NW * WAVE) void gemm_small_kernel(GemmArgs g) {
    constexpr int L = 16, SIDE = T * L, G = 16, CHUNK = U * G;       // tile side; k-values per load, per chunk
    extern __shared__ __align__(16) unsigned char small_lds[];       // [NW - 1][T * T][WAVE] accumulators, then the epilogue's stage
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & (L - 1), q = lane / L;
    const unsigned mt = (unsigned)((g.M + SIDE - 1) / SIDE), tiles = mt * (unsigned)((g.N + SIDE - 1) / SIDE);
    // neighbours along M on one XCD, so that a column of tiles reads its part of B through one L2
    const unsigned id = (blockIdx.x % NUM_XCD) * (gridDim.x / NUM_XCD) + blockIdx.x / NUM_XCD;
    if (id >= tiles) return;
    const int m0 = (int)(id % mt) * SIDE, n0 = (int)(id / mt) * SIDE;
    const int K = g.K, chunks = (K + CHUNK - 1) / CHUNK, whole = K / CHUNK;
    // rows and columns past the matrix: its last one's, whose products are not stored
    const float *pa[T], *pb[T];
#pragma unroll
    for (int t = 0; t < T; t++) {
        pa[t] = g.a + (long long)min(m0 + t * L + j, g.M - 1) * g.lda;
        pb[t] = BT ? g.b + (long long)min(n0 + t * L + j, g.N - 1) * g.ldb : g.b + min(n0 + t * L + j, g.N - 1);
    }

    struct Chunk {
        f32x4 a[U][T], b[U][T];
    };
    auto load = [&](int c, Chunk &x) {
        const int k0 = c * CHUNK + 4 * q;
        if (c < whole) {                                             // uniform
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int k = k0 + u * G;
#pragma unroll
                for (int t = 0; t < T; t++) {
                    x.a[u][t] = *reinterpret_cast<const row_f32x4 *>(pa[t] + k);
                    if (BT) {
                        x.b[u][t] = *reinterpret_cast<const row_f32x4 *>(pb[t] + k);
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; i++) x.b[u][t][i] = pb[t][(long long)(k + i) * g.ldb];
                    }
                }
            }
        } else {                                                     // the last of K: zeros past its end
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int k = k0 + u * G;
#pragma unroll
                for (int t = 0; t < T; t++)
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const bool in = k + i < K;
                        x.a[u][t][i] = in ? pa[t][k + i] : 0.f;
                        x.b[u][t][i] = in ? (BT ? pb[t][k + i] : pb[t][(long long)(k + i) * g.ldb]) : 0.f;
                    }
            }
        }
    };
    f32x4 sum[ACC][T][T];                                            // (four: of the k-values that are 0, 1, 2, 3 modulo four)
#pragma unroll
    for (int i = 0; i < ACC * T * T; i++) sum[i / (T * T)][i / T % T][i % T] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](const Chunk &x) {
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int r = 0; r < T; r++)
#pragma unroll
                    for (int c = 0; c < T; c++) sum[i % ACC][r][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.a[u][r][i], x.b[u][c][i], sum[i % ACC][r][c], 0, 0, 0);
    };
    if (wave < chunks) {
        Chunk x, y;
        load(wave, x);
        int c = wave;
        for (; c + NW < chunks; c += NW) {
            load(c + NW, y);
            __builtin_amdgcn_sched_barrier(0);
            multiply(x);
            x = y;
        }
        multiply(x);
    }
    f32x4 acc[T][T];
#pragma unroll
    for (int i = 0; i < T * T; i++) {
        const int r = i / T, c = i % T;
        if constexpr (ACC == 4) acc[r][c] = (sum[0][r][c] + sum[1][r][c]) + (sum[2][r][c] + sum[3][r][c]);
        else acc[r][c] = sum[0][r][c];
    }
    f32x4 *const part = reinterpret_cast<f32x4 *>(small_lds);
    if (wave) {
#pragma unroll
        for (int i = 0; i < T * T; i++) part[((wave - 1) * T * T + i) * WAVE + lane] = acc[i / T][i % T];
    }
    __syncthreads();
    if (wave) return;
#pragma unroll
    for (int w = 1; w < NW; w++)
#pragma unroll
        for (int i = 0; i < T * T; i++) acc[i / T][i % T] += part[((w - 1) * T * T + i) * WAVE + lane];
    gemm_finish<EPI, L, 1>(g, acc, m0, n0, small_lds + (NW - 1) * T * T * WAVE * sizeof(f32x4));
}

template <bool BT, int T, int U, int NW, int ACC, int EPI>
static void launch_small_as(const GemmArgs &g, long long tiles, hipStream_t st) {
    const size_t lds = (size_t)(NW - 1) * T * T * 256 * sizeof(float) + (EPI == 2 ? gemm_stage_bytes(1) : 0);
    hipLaunchKernelGGL((gemm_small_kernel<BT, T, U, NW, ACC, EPI>), dim3((unsigned)((tiles + NUM_XCD - 1) / NUM_XCD * NUM_XCD)), dim3(NW * WAVE), lds, st, g);
}
// us by form (side 16 with one, four and eight waves; side 32): 1000 x 300 -> 200, 819 squares of 16, 6.5 7.4 7.4 7.1;   130 x 1920 -> 1383, 783, 28.8 29.3
// 28.4 18.4;   17 x 352 -> 6317, 790, 9.0 9.0 9.5 6.7;   310 x 320 -> 576, 720, 6.5 6.4 7.8 7.7;   497 x 1568 -> 232, 480, 17.8 14.9 15.0 16.1;   3000 x 100 -> 50, 752,
// 4.1 4.2 5.3 5.5;   64 x 784 -> 512, 128, 9.0 5.3 5.1 9.9;   64 x 964 x 23, 8, 13.2 6.2 5.6 11.6.
template <bool BT, int EPI>
static void launch_small_epi(const GemmArgs &g, long long tiles, hipStream_t st) {
    const long long t16 = gemm_small_squares(g.M, g.N, 16);
    if (t16 > 840 || (t16 > 600 && g.K > 340)) {
        if (g.K < 640 || tiles > 102) launch_small_as<BT, 2, 2, 4, 1, EPI>(g, gemm_small_squares(g.M, g.N, 32), st);
        else launch_small_as<BT, 2, 2, 4, 4, EPI>(g, gemm_small_squares(g.M, g.N, 32), st);
    } else if (g.K <= 64) launch_small_as<BT, 1, 4, 1, 1, EPI>(g, t16, st);
    else if (g.K <= 256 || t16 > 384) launch_small_as<BT, 1, 4, 4, 4, EPI>(g, t16, st);
    else launch_small_as<BT, 1, 4, 8, 4, EPI>(g, t16, st);
}

// `tiles`: of the fp32 tiles (linear.hip)
bool gemm_small_takes(const GemmArgs &g, bool b_transposed, long long tiles) {
    if (g.bm) return false;                                          // (a caller that names the tile height keeps it)
    const bool whole = g.vec_a && g.vec_b && g.K % 32 == 0 && (b_transposed || g.N % 4 == 0);
    return gemm_small_pays(g.M, g.N, g.K, b_transposed, whole, tiles);
}
hipError_t launch_gemm_small(const GemmArgs &g, bool b_transposed, long long tiles, hipStream_t st) {
    if (!b_transposed) launch_small_epi<false, 0>(g, tiles, st);
    else if (g.cand) launch_small_epi<true, 2>(g, tiles, st);
    else if (g.best) launch_small_epi<true, 1>(g, tiles, st);
    else launch_small_epi<true, 0>(g, tiles, st);
    return hipGetLastError();
}

}  // namespace born
