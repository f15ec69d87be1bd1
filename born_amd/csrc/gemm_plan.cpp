// Host side of the large products (gemm_split.hip): which go there, in which tiles and slices.
#include "gemm_plan.h"

#include <algorithm>
#include <cmath>

namespace born {

// Whether the product goes to the bf16 matrix cores.  They do an fp32 product's work about twice as fast,
// after a launch that packs the left operand: below about 3 GFLOP the fp32 tiles, finer and split along K, are level
// (64 x 4096 -> 4096, 2.1 GFLOP: 33 us against 28; 1024^3 24 against 32; 128 x 4096 -> 4096, 4.3: 72 against 41; 200 x 1056 ->
// 8272, 3.5: 72 against 45); a batch of up to 32 rows is bound by reading the weights (32 x 4096 -> 32000: 118 against 130 us).
// The kernel's loads reach 32 rows of the weights by 32-bit byte offsets: 31 ldb + 31 values of four bytes, and 32 bytes, stay below
// 2^32 up to a pitch of 2^25.
bool gemm_split_pays(int M, int N, int K, long long ldb) {
    return M > 32 && ldb <= (1ll << 25) && 2.0 * (double)M * (double)N * (double)K >= 3e9;
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

// Tile and slices of K with the least expected time: rounds of tiles over the CUs, each with about 8 us to fill and drain;
// slices write and re-read partial products (about 4 TB/s) and cost one more launch.  Measured against the choice on
// twenty shapes: within 15 % of the best of all of them (256 x 4096 -> 4096: 128 x 128 in four slices 61 us, 128 us unsplit,
// 425 us as 256 x 256; 300 x 2528 -> 21539: 128 x 256 179 us, 64 x 128 212, 256 x 256 288).
SplitPlan gemm_split_plan(int M, int N, int K) {
    constexpr float CUS = 256.f;
    SplitPlan best = {0, 1};
    float least = INFINITY;
    for (int t = 0; t < 4; t++) {
        const SplitTile &T = SPLIT_TILES[t];
        const float tiles = (float)((M + T.rows - 1) / T.rows) * (float)((N + T.cols - 1) / T.cols);
        for (int slices = 1; slices <= 16 && (slices == 1 || K / slices >= 256); slices *= 2) {
            if (slices > 1 && tiles * slices > 2.f * CUS) break;
            const float wgs = tiles * slices, rounds = std::ceil(wgs / CUS);
            const float share = std::min(1.f, wgs / CUS);
            float us = rounds * ((T.idle_us + (T.busy_us - T.idle_us) * share) * ((float)K / 4096.f) / slices + 8.f);
            if (slices > 1) us += 3.f + (float)M * (float)N * 4.f * (slices + 1) / 4e6f;
            if (us < least) {
                least = us;
                best.tile = t;
                best.slices = slices;
            }
        }
    }
    // whole pairs of groups to a slice, none of them empty
    const int pairs = (K + 2 * SG - 1) / (2 * SG), per = (pairs + best.slices - 1) / best.slices;
    best.slices = (pairs + per - 1) / per;
    best.kslice = per * 2 * SG;
    return best;
}

}  // namespace born
