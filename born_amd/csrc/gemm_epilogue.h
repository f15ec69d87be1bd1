// What the GEMM kernels (linear.hip, gemm_split.hip) do with a tile's results, and the types they share.
#pragma once
#include "dev_common.h"
#include "kernels.h"

namespace born {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int GEMM_THREADS = 256;
constexpr int NUM_XCD = 8;

// What a tile does with its results.  EPI 0: adds the bias and stores them.  EPI 1 (greedy decode fused into
// the LM head): keeps only the largest logit of every row as a packed key, value in the high word, ~column in
// the low word, merged across tiles with a 64-bit atomic max, so the logits are never written.  The key order
// is the reference's argmax (internal/nn/cross_entropy.go:241-251): larger value wins, the lower index on equal
// values (-0 equals +0), a NaN never wins, except at index 0 where the reference returns 0 whatever follows.
__device__ __forceinline__ u64 gemm_argmax_key(float v, int col) {
    if (v != v) return col == 0 ? ~0ull : 0ull;
    v = v == 0.0f ? 0.0f : v;
    return ((u64)ordkey(v) << 32) | (u64)(0xFFFFFFFFu - (u32)col);
}
__device__ __forceinline__ u64 gemm_max_u64(u64 a, u64 b) { return a > b ? a : b; }
// The keys of consecutive rows sit a cache line apart, and a tile first looks at the key it would have to beat:
// the value only ever grows, so a tile that does not beat what it reads (however stale) cannot win, and all but
// the first few tiles of a row skip the atomic.
constexpr int GEMM_BEST_PITCH = LM_BEST_PITCH; // u64 words between the keys of consecutive rows (a 128-byte line each)
__device__ __forceinline__ void gemm_offer_key(u64 *best, int row, u64 key) {
    u64 *p = best + (long long)row * GEMM_BEST_PITCH;
    if (key > __builtin_nontemporal_load(p)) atomicMax(p, key);
}
__device__ __forceinline__ u64 gemm_shfl_xor_u64(u64 x, int o) {
    const u32 lo = (u32)__shfl_xor((int)(u32)x, o, WAVE), hi = (u32)__shfl_xor((int)(u32)(x >> 32), o, WAVE);
    return ((u64)hi << 32) | lo;
}

// EPI 2 (sampling fused into the LM head): every result at or above its row's threshold is appended, value and
// column, to the row's candidate list (one global atomic per candidate: a few per row and tile); the logits are
// never written.  A NaN is never listed.  The counter may run past the list's capacity: the reader sees that.
__device__ __forceinline__ void gemm_offer_candidate(const GemmArgs &g, int row, int col, float v, float thr) {
    if (v >= thr) {
        const unsigned pos = atomicAdd(&g.cand_cnt[(long long)row * LM_CAND_PITCH], 1u);
        if (pos < (unsigned)g.cand_cap) g.cand[(long long)row * g.cand_cap + pos] = make_uint2(__float_as_uint(v), (unsigned)col);
    }
}

// The results of a wave: IB x JB blocks of L x L, L = 32 or 16 as the matrix instruction leaves them - register v of lane
// (c, h), c = lane % L, h = lane / L, is row 8 (v / 4) + 4 h + v % 4, column c of its block.  row0, col0: the wave's first.
// stage: LDS of the workgroup's NW waves for EPI 2, gemm_stage_bytes(NW), 8-byte aligned, that nobody uses any more.
constexpr int GEMM_STAGE = 192;
constexpr int gemm_stage_bytes(int waves) { return waves * GEMM_STAGE * (int)(sizeof(uint2) + sizeof(int)); }
template <int EPI, int L, int NW, typename V, int IB, int JB>
__device__ __forceinline__ void gemm_finish(const GemmArgs &g, const V (&acc)[IB][JB], int row0, int col0, void *stage) {
    constexpr int REGS = L * L / WAVE;
    static_assert(sizeof(V) == REGS * sizeof(float), "block shape");
    const int lane = (int)(threadIdx.x & (WAVE - 1)), c = lane & (L - 1), h = lane / L;
    auto row_of = [&](int i, int v) { return row0 + i * L + (v >> 2) * 8 + h * 4 + (v & 3); };
    if (EPI == 0) {
#pragma unroll
        for (int j = 0; j < JB; j++) {
            const int col = col0 + j * L + c;
            if (col >= g.N) continue;
            const float bias = g.bias ? g.bias[col] : 0.f;
#pragma unroll
            for (int i = 0; i < IB; i++) {
#pragma unroll
                for (int v = 0; v < REGS; v++) {
                    const int row = row_of(i, v);
                    if (row < g.M) {
                        const float sum = acc[i][j][v];
                        g.c[(long long)row * g.ldc + col] = g.bias ? sum + bias : sum;
                    }
                }
            }
        }
    } else if (EPI == 2) {
        // A candidate's place in its row's list costs a global atomic, and one per candidate where it is met would make
        // the wave wait for a memory round trip some forty times.  The wave stages its candidates in LDS instead
        // (ballot + lane rank, no atomics) and then asks for all their places at once.
        constexpr int STAGE = GEMM_STAGE;                            // a 64 x 64 block of C yields about 70
        uint2 *const vc = reinterpret_cast<uint2 *>(stage) + (threadIdx.x >> 6) * STAGE;
        int *const rw = reinterpret_cast<int *>(reinterpret_cast<uint2 *>(stage) + NW * STAGE) + (threadIdx.x >> 6) * STAGE;
        u32 count = 0;                                               // wave-uniform
        float bias[JB];
#pragma unroll
        for (int j = 0; j < JB; j++) {
            const int col = col0 + j * L + c;
            bias[j] = (g.bias && col < g.N) ? g.bias[col] : 0.f;
        }
#pragma unroll
        for (int i = 0; i < IB; i++) {
#pragma unroll
            for (int v = 0; v < REGS; v++) {
                const int row = row_of(i, v);
                const float thr = row < g.M ? g.thr[row] : INFINITY;
#pragma unroll
                for (int j = 0; j < JB; j++) {
                    const int col = col0 + j * L + c;
                    const float sum = acc[i][j][v];
                    const float val = g.bias ? sum + bias[j] : sum;
                    const bool pass = col < g.N && row < g.M && val >= thr;   // a NaN never passes
                    const u64 m = __ballot(pass);
                    if (m) {                                         // wave-uniform
                        if (pass) {
                            const u32 pos = count + __builtin_amdgcn_mbcnt_hi((u32)(m >> 32), __builtin_amdgcn_mbcnt_lo((u32)m, 0u));
                            if (pos < (u32)STAGE) {
                                vc[pos] = make_uint2(__float_as_uint(val), (unsigned)col);
                                rw[pos] = row;
                            } else {
                                gemm_offer_candidate(g, row, col, val, thr);   // the stage is full: straight to the list
                            }
                        }
                        count += (u32)__popcll(m);
                    }
                }
            }
        }
        const int staged = (int)min(count, (u32)STAGE);
        for (int e = lane; e < staged; e += WAVE) {                  // (the wave's own LDS writes are visible to it in order)
            const int row = rw[e];
            const unsigned pos = atomicAdd(&g.cand_cnt[(long long)row * LM_CAND_PITCH], 1u);
            if (pos < (unsigned)g.cand_cap) g.cand[(long long)row * g.cand_cap + pos] = vc[e];
        }
    } else {
        float bias[JB];
#pragma unroll
        for (int j = 0; j < JB; j++) {
            const int col = col0 + j * L + c;
            bias[j] = (g.bias && col < g.N) ? g.bias[col] : 0.f;
        }
#pragma unroll
        for (int i = 0; i < IB; i++) {
#pragma unroll
            for (int v = 0; v < REGS; v++) {
                if (row0 + i * L + (v >> 2) * 8 + (v & 3) >= g.M) continue;   // past the batch for every h: wave-uniform
                u64 key = 0ull;
#pragma unroll
                for (int j = 0; j < JB; j++) {
                    const int col = col0 + j * L + c;
                    const float sum = acc[i][j][v];
                    if (col < g.N) key = gemm_max_u64(key, gemm_argmax_key(g.bias ? sum + bias[j] : sum, col));
                }
#pragma unroll
                for (int o = L / 2; o > 0; o >>= 1) key = gemm_max_u64(key, gemm_shfl_xor_u64(key, o));   // the L lanes of this h
                const int row = row_of(i, v);
                if (c == 0 && row < g.M && key) gemm_offer_key(g.best, row, key);
            }
        }
    }
}

}  // namespace born
