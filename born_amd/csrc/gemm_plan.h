// Which products go to the bf16 matrix cores (gemm_split.hip), in which tiles and slices: host decisions without HIP.
#pragma once
#include <cstddef>

namespace born {

constexpr int SG = 32;                        // k-values of a group (two matrix instructions deep)
constexpr int SG_BYTES = 6 * 1024;            // packed bytes of a group and a block of 32 rows
constexpr int PACK_GROUPS = 4;                // groups a workgroup of the pack handles

// A plan: which of the tiles, how many slices of K (kslice values each).
struct SplitPlan {
    int tile, slices, kslice;
};
bool gemm_split_pays(int M, int N, int K, long long ldb);
SplitPlan gemm_split_plan(int M, int N, int K);
size_t gemm_split_workspace(int M, int K);    // bytes of the packed operand and its flags, a multiple of 256

}  // namespace born
