// Host side of the large products (gemm_split.hip): which go there, in which tiles and slices.
#include "gemm_plan.h"

#include <algorithm>
#include <cmath>

namespace born {

// Whether the product goes to the bf16 matrix cores.  They do an fp32 product's work about twice as fast,
// after a launch that packs the left operand: below about 3 GFLOP the fp32 tiles, finer and split along K, are level
// (64 x 4096 -> 4096, 2.1 GFLOP: 33 us against 28; 1024^3 24 against 32; 128 x 4096 -> 4096, 4.3: 72 against 41; 200 x 1056 ->
// 8272, 3.5: 72 against 45); a batch of up to 32 rows is bound by reading the weights (32 x 4096 -> 32000: 118 against 130 us).
// A sum of fewer than a dozen terms is more accurate on the fp32 tiles (gemm_split.hip), so K is 16 at least.
// The kernel's loads reach 32 rows of the weights by 32-bit byte offsets: 31 ldb + 31 values of four bytes, and 32 bytes, stay below
// 2^32 up to a pitch of 2^25.
bool gemm_split_pays(int M, int N, int K, long long ldb) {
    return M > 32 && K >= 16 && ldb <= (1ll << 25) && 2.0 * (double)M * (double)N * (double)K >= 3e9;
}

size_t gemm_split_workspace(int M, int K) {
    const size_t ng = (size_t)(K + 2 * SG - 1) / (2 * SG) * 2, mb = (size_t)(M + 31) / 32;
    const size_t bytes = ng * mb * SG_BYTES + 8 * SG_BYTES + mb * ((ng + PACK_GROUPS - 1) / PACK_GROUPS) * 2 * sizeof(unsigned);   // (8 blocks: the last tile's copy may run on)
    return (bytes + 255) / 256 * 256;
}

// The four tiles, and what one of them takes at K = 4096 on a part that is nearly idle and on one where every CU has one
// (power: the clock falls from 2.4 to about 1.9 GHz), in microseconds.
//   64 x 128   four waves' columns twice along K          70 .. 121   decode batches: no matrix work for padding
//   128 x 128  four waves' columns twice along K         120 .. 180   few columns: tiles for all CUs
//   128 x 256  eight waves' columns                      222 .. 317
//   256 x 256  eight waves' columns                      405 .. 532   the most products per byte moved through LDS
struct SplitTile {
    int rows, cols;
    float idle_us, busy_us;
};
constexpr SplitTile SPLIT_TILES[4] = {{64, 128, 70.f, 121.f}, {128, 128, 120.f, 180.f}, {128, 256, 222.f, 317.f}, {256, 256, 405.f, 532.f}};

size_t gemm_split_bytes(const SplitPlan &p, int rows, int N, int K) {
    return gemm_split_workspace(rows, K) + (p.slices > 1 ? (size_t)p.slices * (size_t)rows * (size_t)N * sizeof(float) : 0);
}

// Tile, slices of K and rows at a time with the least expected time, among those whose packed operand and partial products fit the
// workspace: rounds of tiles over the CUs, each with about 8 us to fill and drain; slices write and re-read partial products
// (about 4 TB/s) and cost one more launch; a product whose rows do not fit at once is as many products, each with its own
// launches.  Measured against the choice on twenty shapes that fit at once: within 15 % of the best of all of them (256 x 4096
// -> 4096: 128 x 128 in four slices 61 us, 128 us unsplit, 425 us as 256 x 256; 300 x 2528 -> 21539: 128 x 256 179 us, 64 x
// 128 212, 256 x 256 288).  A choice that would not fit gives way to one that does (us, the fp32 tiles before it): 512 x 4096 -> 4096
// 94 (135), 1024 159 (260), 2048 281 (500), 256 x 4096 -> 8192 92 (135), 512 x 14336 -> 4096 298 (456), 2900 x 4096 -> 2600 in two
// parts 303 (488).
// rows = 0: the fp32 tiles have it.  Nothing fits beyond K = 174 000, where 64 packed rows are more than the workspace; and in parts a
// product has to beat what the fp32 tiles reach at their best, 135 TFLOP/s (4096 x 16384 -> 1024, a long K in eleven parts: 1089 us
// against 1009; 1900 x 8192 -> 130: 96 against 82).
SplitPlan gemm_split_plan(int M, int N, int K) {
    constexpr float CUS = 256.f;
    const long long pairs = ((long long)K + 2 * SG - 1) / (2 * SG);  // of groups
    SplitPlan best = {0, 1, 0, 0};
    float least = INFINITY;
    const float fp32_us = 2.f * (float)M * (float)N * (float)K / 135e6f;
    for (int t = 0; t < 4; t++) {
        const SplitTile &T = SPLIT_TILES[t];
        for (int want = 1; want <= 16 && (want == 1 || K / want >= 256); want *= 2) {
            // whole pairs of groups to a slice, none of them empty
            const long long per = (pairs + want - 1) / want;
            const int slices = (int)((pairs + per - 1) / per);
            // rows at a time: as many tiles' as fit, shared out evenly
            const double block = (double)(2 * pairs * SG_BYTES + (2 * pairs + PACK_GROUPS - 1) / PACK_GROUPS * 8) +
                                 (slices > 1 ? 32.0 * 4.0 * slices * (double)N : 0.0);
            const long long fit = (long long)((double)(GEMM_WS_MAX - 8 * SG_BYTES - 256) / block) * 32;
            long long rows = M;
            if (fit < M) {
                const long long whole = fit / T.rows * T.rows;
                if (whole == 0) continue;
                const long long chunks = (M + whole - 1) / whole;
                rows = ((M + chunks - 1) / chunks + T.rows - 1) / T.rows * T.rows;
            }
            const auto tiles = [&](long long m) { return (float)((m + T.rows - 1) / T.rows) * (float)(((long long)N + T.cols - 1) / T.cols); };
            if (slices > 1 && tiles(rows) * want > 2.f * CUS) continue;
            const auto time = [&](long long m) {
                const float wgs = tiles(m) * want, rounds = std::ceil(wgs / CUS);
                const float share = std::min(1.f, wgs / CUS);
                float us = rounds * ((T.idle_us + (T.busy_us - T.idle_us) * share) * ((float)K / 4096.f) / want + 8.f);
                if (slices > 1) us += 3.f + (float)m * (float)N * 4.f * (want + 1) / 4e6f;
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

}  // namespace born
