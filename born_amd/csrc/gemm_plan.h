// Which products go to the 16-bit matrix cores (gemm_split.hip), in which tiles and slices, and which to the kernel of small ones (gemm_small.hip):
// host decisions without HIP.
#pragma once
#include <cstddef>

namespace born {

constexpr int SG = 32;                        // k-values of a group (two matrix instructions deep)
constexpr int SG_BYTES = 6 * 1024;            // packed bytes of a group and a block of 32 rows, in three parts (two of fp16: 4 KiB, and 2 KiB of what they leave)
constexpr int PACK_GROUPS = 4;                // groups a workgroup of the pack handles

// The workspace of a stream (linear.hip): the packed operand and the partial products of the slices of K.
constexpr size_t GEMM_WS_MAX = (size_t)64 << 20, GEMM_WS_MIN = (size_t)8 << 20;

// A plan: which of the tiles, how many slices of K (kslice values each), how many rows at a time (M, or a multiple of the
// tile's height; 0 where the fp32 tiles have the product after all).
struct SplitPlan {
    int tile, slices, kslice, rows;
};
int gemm_split_parts(int K);                  // of each operand's values: two of fp16, or three of bf16
bool gemm_split_pays(int M, int N, int K, long long ldb);
SplitPlan gemm_split_plan(int M, int N, int K);
size_t gemm_split_workspace(int M, int K);    // bytes of the packed operand and its flags, a multiple of 256
size_t gemm_split_bytes(const SplitPlan &p, int rows, int N, int K);   // .. and of the partial products behind it

inline long long gemm_small_squares(long long M, long long N, int side) { return ((M + side - 1) / side) * ((N + side - 1) / side); }
bool gemm_small_pays(int M, int N, int K, bool b_transposed, bool whole, long long tiles);

}  // namespace born
