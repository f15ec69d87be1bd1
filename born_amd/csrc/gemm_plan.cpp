// Host side of the products: which large ones go to gemm_split.hip, in which tiles and slices, and which small ones to gemm_small.hip.
#include "gemm_plan.h"

#include <algorithm>
#include <cmath>

namespace born {

// Whether the product goes to the 16-bit matrix cores.  They do an fp32 product's work two to three times as fast,
// after a launch that packs the left operand: below about 3 GFLOP the fp32 tiles, finer and split along K, are level (us, theirs
// first: 64 x 4096 -> 4096, 2.1 GFLOP, 30 31; 1024^3 23 28; 64 x 1024 -> 16000 24 28; but 256 x 2048 -> 2048 38 25; above, 128 x 4096 -> 4096 72 35,
// 200 x 1056 -> 8272 72 35).  Up to 32 rows are bound by reading the weights, which these kernels do better down a long K (17 x 4096 -> 32000
// 120 97, 32 118 90, 32 x 4096 -> 128256 375 361; 32 x 512 -> 100000 46 63, 20 x 1024 -> 50000 41 49); up to 16 the fp32 tiles read as fast.
// A sum of fewer than a dozen terms is more accurate on the fp32 tiles (gemm_split.hip), so K is 16 at least.
// The kernel's loads reach 32 rows of the weights by 32-bit byte offsets: 31 ldb + 31 values of four bytes, and 32 bytes, stay below
// 2^32 up to a pitch of 2^25.
bool gemm_split_pays(int M, int N, int K, long long ldb) {
    return (M > 32 ? K >= 16 : M > 16 && K >= 2048) && ldb <= (1ll << 25) && 2.0 * (double)M * (double)N * (double)K >= 3e9;
}

// Two fp16 parts lose 2^-23.7 of a product, root mean square, and round a sum a third as often as three bf16 parts; from a K of 256 on the sum is closer
// to fp64 for it (K = 256 1.18e-7 against 1.55e-7, normal operands; below, what is lost and what is gained come level), and it
// is half the matrix instructions (gemm_split.hip).
int gemm_split_parts(int K) { return K >= 256 ? 2 : 3; }

size_t gemm_split_workspace(int M, int K) {
    const size_t ng = (size_t)(K + 2 * SG - 1) / (2 * SG) * 2, mb = (size_t)(M + 31) / 32;
    const size_t bytes = ng * mb * SG_BYTES + 8 * SG_BYTES + mb * ((ng + PACK_GROUPS - 1) / PACK_GROUPS) * 2 * sizeof(unsigned) + mb * 32 * (4 * sizeof(int) + 1);   // (8 blocks: the last tile's copy may run on)
    return (bytes + 255) / 256 * 256;
}

// The four tiles, and what one of them takes at K = 4096 on a part that is nearly idle and on one where every CU has one
// (power: the clock falls), in microseconds; what a round of tiles takes besides, to fill and drain; and what slices of K take: a launch, and
// writing and reading the partial products again.  Two parts, then three: two parts' fitted to 44 shapes in every tile and up to 16 slices (the
// choice is within 1 % of the best of them on average, 19 % at worst: 88 x 2144 -> 11475).  Three parts have a K below 256, so they are not sliced; their
// times are those of a K of 4096 in proportion.
//   64 x 128   four waves' columns twice along K    decode batches: no matrix work for padding
//   128 x 128  four waves' columns twice along K    few columns: tiles for all CUs
//   128 x 256  eight waves' columns
//   256 x 256  eight waves' columns                 the most products per byte moved through LDS
constexpr int SPLIT_TILES = 4, SPLIT_ROWS[SPLIT_TILES] = {64, 128, 128, 256}, SPLIT_COLS[SPLIT_TILES] = {128, 128, 256, 256};
struct SplitTimes {
    float idle_us[SPLIT_TILES], busy_us[SPLIT_TILES], round_us;
};
constexpr SplitTimes SPLIT_TIMES[2] = {{{44.f, 80.f, 170.f, 198.f}, {66.f, 114.f, 208.f, 390.f}, 4.f}, {{70.f, 120.f, 222.f, 405.f}, {121.f, 180.f, 317.f, 532.f}, 8.f}};
constexpr float SLICES_US = 0.2f, SLICES_BYTES_PER_US = 3.3e6f;

size_t gemm_split_bytes(const SplitPlan &p, int rows, int N, int K) {
    return gemm_split_workspace(rows, K) + (p.slices > 1 ? (size_t)p.slices * (size_t)rows * (size_t)N * sizeof(float) : 0);
}

// Tile, slices of K and rows at a time with the least expected time, among those whose packed operand and partial products fit the
// workspace: rounds of tiles over the CUs, each with 4 us (three parts 8) to fill and drain; slices write and re-read partial products
// and cost one more launch; a product whose rows do not fit at once is as many products, each with its own
// launches.  (256 x 4096 -> 4096: 128 x 128 in four slices 48 us, 128 x 256 in eight 51; 300 x 2528 -> 21539: 128 x 256 145 us, 64 x
// 128 172, 256 x 256 191.)  A choice that would not fit gives way to one that does (us, the fp32 tiles): 512 x 4096 -> 4096
// 75 (135), 1024 124 (260), 2048 217 (500), 256 x 4096 -> 8192 73 (135), 512 x 14336 -> 4096 219 (456), 2900 x 4096 -> 2600 in two
// parts 242 (488).
// rows = 0: the fp32 tiles have it.  Nothing fits beyond K = 174 000, where 64 packed rows are more than the workspace; and in parts a
// product has to beat what the fp32 tiles reach at their best, 135 TFLOP/s (4096 x 16384 -> 1024, a long K in eleven parts: 1089 us
// against 1009; 1900 x 8192 -> 130: 96 against 82).
SplitPlan gemm_split_plan(int M, int N, int K) {
    constexpr float CUS = 256.f;
    const long long pairs = ((long long)K + 2 * SG - 1) / (2 * SG);  // of groups
    SplitPlan best = {0, 1, 0, 0};
    float least = INFINITY;
    const float fp32_us = 2.f * (float)M * (float)N * (float)K / 135e6f;
    const SplitTimes &T = SPLIT_TIMES[gemm_split_parts(K) - 2];
    for (int t = 0; t < SPLIT_TILES; t++) {
        const int tile_rows = SPLIT_ROWS[t], tile_cols = SPLIT_COLS[t];
        for (int want = 1; want <= 16 && (want == 1 || K / want >= 256); want *= 2) {
            // whole pairs of groups to a slice, none of them empty
            const long long per = (pairs + want - 1) / want;
            const int slices = (int)((pairs + per - 1) / per);
            // rows at a time: as many tiles' as fit, shared out evenly
            const double block = (double)(2 * pairs * SG_BYTES + (2 * pairs + PACK_GROUPS - 1) / PACK_GROUPS * 8 + 32 * 17) +
                                 (slices > 1 ? 32.0 * 4.0 * slices * (double)N : 0.0);
            const long long fit = (long long)((double)(GEMM_WS_MAX - 8 * SG_BYTES - 256) / block) * 32;
            long long rows = M;
            if (fit < M) {
                const long long whole = fit / tile_rows * tile_rows;
                if (whole == 0) continue;
                const long long chunks = (M + whole - 1) / whole;
                rows = ((M + chunks - 1) / chunks + tile_rows - 1) / tile_rows * tile_rows;
            }
            const auto tiles = [&](long long m) { return (float)((m + tile_rows - 1) / tile_rows) * (float)(((long long)N + tile_cols - 1) / tile_cols); };
            if (slices > 1 && tiles(rows) * want > 2.f * CUS) continue;
            const auto time = [&](long long m) {
                const float wgs = tiles(m) * want, rounds = std::ceil(wgs / CUS);
                const float share = std::min(1.f, wgs / CUS);
                float us = rounds * ((T.idle_us[t] + (T.busy_us[t] - T.idle_us[t]) * share) * ((float)K / 4096.f) / want + T.round_us);
                if (slices > 1) us += SLICES_US + (float)m * (float)N * 4.f * (want + 1) / SLICES_BYTES_PER_US;
                return us;
            };
            const long long chunks = (M + rows - 1) / rows, last = M - (chunks - 1) * rows;
            const float us = (float)(chunks - 1) * (time(rows) + 6.f) + time(last);
            if (us < least && (chunks == 1 || us < fp32_us)) {
                least = us;
                best = SplitPlan{t, slices, (int)(per * 2 * SG), (int)rows};
            }
        }
    }
    return best;
}

// ---- which small products go to gemm_small.hip, not to the fp32 tiles (linear.hip)
// Where the tiles' loads are guarded ones.  us, tiles and here, linear and then matmul:
//   a long K and few squares, a CU to each: the tiles' slices are on more of them
//     1 square   3211 13.5 11.1, 16.9 10.8;   4097 15.2 16.7, 19.3 12.6;   8193 21.2 30.3, 28.2 21.6;   24 001 43 83, 61 55;   40 001 66 137, 96 94
//     4          6001 17.9 16.7, 24.9 19.0;   8193 21.8 26.5, 31.3 23.4;   24 001 44 71, 68 57
//     21         8193 31.2 30.8, 30.9 24.6;   12 001 39.6 43.7, 38.9 42.5
//     42         12 001 43.8 44.6, 44.4 44.6;   20 001 64 71, 65 71;   126: 8193 36.2 30.9, 31.0 28.4;   169: 8193 48 31, 35 31, 12 001 67 45, 45 43
//     288        4097 33.2 31.3, 34.7 32.5;   6001 40.5 38.7, 41.8 45.7 (the CUs' second round);   425: 4097 38.9 31.4, 30.6 30.9
//     up to four rows, which are few lines here: 3 x 100 003 -> 10 148 138, 240 202, -> 252 257 176, 222 209, -> 700 282 206, 228 303;   3 x 30 001 -> 700 87 57, 75 73;   2 x 15 391 -> 18 30 36
//     few columns of many rows, of which a tile wastes most: 911 x 19 590 -> 17 73 52, 92 56, 3415 x 35 508 -> 2 361 94, 502 108;   768 x 30 001 -> 9 97 65, 132 74
//   large results of a short K, which the tiles store in whole lines where rows are a multiple of 16 bytes
//     250 000 squares  8000 x 3 -> 8000 157 166, 143 198;   64 000: 4096 x 7 -> 4000 43 47, 39 56;   47 000: 3000 x 7 -> 4000 41 36, 37 43
//     16 000 4096 x 20 -> 1000 18.8 17.2, 17.6 19.4;   32 000: 4096 x 50 -> 2000 33 34, 28 37;   8192: 4096 x 204 -> 500 20.4 25.2, 21.1 22.8, half the tiles' error (above 32 values here it is
//     smaller than theirs)
//     rows of odd length 16 000 1000 x 7 -> 4001 20.0 15.6, 18.5 18.2;   37 500 200 000 x 7 -> 33 68 40, 66 50
static bool small_pays_guarded(int M, int N, int K, bool b_transposed) {
    const long long squares = gemm_small_squares(M, N, 16);
    if ((double)M * (double)N * (double)K > 5e8) return false;
    if (N > 32 || M < 768) {
        int k_max;
        if (M <= 4 && (!b_transposed || squares == 1 || squares > 3)) k_max = b_transposed || squares <= 16 ? 131072 : 32768;
        else if (b_transposed) k_max = squares < 4 ? 3584 : squares < 21 ? 6144 : squares < 42 ? 8448 : squares <= 256 ? 12288 : 4352;
        else k_max = squares < 16 ? 24576 : squares <= 256 ? 10240 : 4352;
        if (K > k_max) return false;
    }
    return N % 4 || squares <= (b_transposed ? 48000 : K > 32 ? 16384 : 3072);
}
// `tiles`: of the fp32 tiles.  whole: their loads need no guard, K a multiple of 32 and all aligned.  us, theirs and here:
//   columns that fill half a tile or less  4096 x 1024 -> 64 21.1 13.1, 2048 x 8192 -> 16 45 31, 512 x 4096 -> 64 16.8 17.0, 512 x 8192 -> 64 21.8 30.6, 1024 x 4096 -> 64 21.2 17.1, 1100 x 4096 -> 64
//                     21.9 30.6, 1024 x 8192 -> 32 29.4 30.6
//   more than 128 tiles, which are left unsliced  2048 x 128 -> 512 7.0 8.5, 7 x 320 -> 21 263 8.1 10.6
//   few squares and a long K, where slices put more CUs to work  16 x 4096 -> 1000 13.2 16.8;   128 squares: 3072 13.2 13.3, 4096 15.1 16.7;   148: 22 x 4096 -> 1170 16.0 16.7;   183: 6 x 4096 -> 2928
//                     17.1 13.5;   250: 14 x 3616 -> 4000 18.6 15.4
//   257 to 384, a second round of CUs  17 x 960 -> 2594 10.5 9.5, 12 x 1408 -> 4456 12.4 12.0, 17 x 1440 -> 2524 11.8 14.0, 32 x 1888 -> 2076 14.0 17.1, 18 x 3808 -> 2301 19.5 30.0;   more than 32 rows:
//                     64 x 1408 -> 1410 15.6 12.9, 40 x 1664 -> 1604 15.6 14.4, 64 x 2016 -> 1108 14.6 17.9
//   385 to 512, four waves each  128 x 1472 -> 901 17.1 12.9, 17 x 1792 -> 3701 15.3 15.1, 24 x 1888 -> 3100 16.3 16.8, 20 x 2112 -> 3648 16.8 17.9
//   above             20 x 960 -> 4587 12.2 12.9, 17 x 1056 -> 4696 12.5 15.3, 100 x 1504 -> 1329 17.7 19.5;   from 600 on in squares of 32: 200 x 1280 -> 766 17.0 13.8, 17 x 1568 -> 5009 15.6 16.2;   which up to 16
//                     rows fill half: 6 x 384 -> 8728 8.0 5.8, 6 x 672 -> 10 967 11.3 12.1, 8 x 1568 -> 11 388 18.0 23.2
bool gemm_small_pays(int M, int N, int K, bool b_transposed, bool whole, long long tiles) {
    if (!whole) return small_pays_guarded(M, N, K, b_transposed);
    const double products = (double)M * (double)N * (double)K;
    const long long squares = gemm_small_squares(M, N, 16);
    if (N <= 64 && products <= 3e8) return K <= 2048 || (M >= 1024 && squares >= 128 && (N <= 16 || (K <= 4096 && squares <= 256)));
    if (tiles >= 128 || products > 2.1e8) return false;
    if (squares <= 256) return K <= (squares < 128 ? 2048 : squares < 144 ? 3072 : 4096);
    if (squares <= 384) return K <= (M > 32 ? 1700 : 1400);
    if (squares <= 512) return K <= 2048;
    return K <= (M <= 16 ? 640 : squares <= 600 ? 1000 : 1700);
}

}  // namespace born
