// The large products on the bf16 matrix cores.
//
// The fp32 matrix pipe of this part runs at 157 TFLOP/s, the bf16 pipe at 2.5 PFLOP/s.  An fp32 number is the exact sum
// of three bf16 numbers (24 significand bits = 3 x 8: each part is the rounded rest of the ones before; the method of Henry, Tang
// and Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype For Higher-Precision Computations", 2019), so a product
// is nine bf16 products, each exact in fp32.  The six largest are computed.  With a = a1 + a2 + a3 the parts fall by 2^-8 and 2^-17
// of a at least, so what is left out (a2 b3, a3 b2, a3 b3) is at most about 2^-24 |a b|, half an ulp, and 2^-27 as a root mean square.
// Accumulation stays in fp32, in the matrix unit's accumulators, 32 k-values to an addition where the fp32 form has two.
//
// Error against fp64, 2-norm, measured beside the fp32 tiles': sums of 12 terms and more never larger, whatever their signs and
// magnitudes (normal operands 0.45 of it at K = 16, 0.64 at 64, 0.59 at 1024, 0.94 at 4096; positive ones 0.56, 0.64, 0.39, 0.87;
// equal significands with the largest omission 1.00); sums of one to four terms that are not zero larger by up to 1.6, one such term
// by up to 2.8 half-ulps where the fp32 unit rounds it once.  K below 16 is therefore not taken (gemm_split_pays); a longer sum of
// which all but a few terms are zero is, and has that error (exactly 0 where a factor is a power of two, as in a selection of rows).
//
//   * Pack: the left operand [M,K] (activations) is split once per call into a workspace laid out as the matrix
//     instructions read it: per group of 32 k-values and block of 32 rows six 1 KiB operands (two halves of 16 rows x three
//     parts), each the 16 bytes of 64 lanes in lane order.  A stage of a tile is then a linear copy into LDS and every
//     operand read of 16 bytes per lane is linear too: no bank conflicts, no address arithmetic.
//   * The right operand (weights) belongs to one wave each: a wave owns 32 of its rows (columns of C) alone, copies them
//     straight into LDS of its own, reads what its lanes feed to the matrix unit and splits it in registers (5.5 vector
//     instructions per value, between the matrix instructions of the group before).
//   * v_mfma_f32_16x16x32_bf16 rather than 32x32x16: at full rate this part is limited by power, and on random operands the
//     16 x 16 form sustains 1.9 PFLOP/s where the 32 x 32 form sustains 1.7.
//   * C tiles are 32 IB x 32 NW: IB blocks of 32 rows per wave, NW waves side by side.
//
// Bound by power: at 256 x 4096 -> 128256 the matrix pipes are busy in 76 % of the cycles at a clock that has fallen from 2.4 to
// 1.9 GHz, and a bare loop of the instruction on random operands does no more than 1.9 PFLOP/s.  Measured against the fp32 tiles of linear.hip (us): 256 x 4096 -> 128256 2060 -> 1065 (253 TFLOP/s of
// fp32 work, 1.5 PFLOP/s of bf16), 128 x 4096 -> 32000 280 -> 174, 64 x 4096 -> 32000 160 -> 126, 2048^3 137 -> 88.
//
// Values outside what bf16 parts can hold - an infinity or NaN anywhere, magnitudes below 2^-100 whose third part would
// be lost - are noticed at the end (by non-finite results; by flags the pack keeps of its operand; by a scan of the
// weights where either those flags or a result near zero make their magnitudes matter), and the wave recomputes its
// block with fp32 matrix instructions (gemm_recompute), so such operands give what they always gave.
#include "gemm_epilogue.h"
#include "gemm_plan.h"

namespace born {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef u32 u32x4 __attribute__((ext_vector_type(4)));

constexpr float SPLIT_BIG = 0x1p30f;          // against a partner up to this the loss stays below 2^-96 per product
constexpr float SPLIT_SMALL_RESULT = 0x1p-60f;   // .. which a result at or above this does not feel

// The three parts of two numbers, as packed pairs of bf16.
__device__ __forceinline__ void split_pair(float x, float y, u32 &p1, u32 &p2, u32 &p3) {
    const f32x2 v = {x, y};
    p1 = __builtin_bit_cast(u32, __builtin_convertvector(v, bf16x2));
    const f32x2 r = {x - __uint_as_float(p1 << 16), y - __uint_as_float(p1 & 0xFFFF0000u)};
    p2 = __builtin_bit_cast(u32, __builtin_convertvector(r, bf16x2));
    const f32x2 q = {r.x - __uint_as_float(p2 << 16), r.y - __uint_as_float(p2 & 0xFFFF0000u)};
    p3 = __builtin_bit_cast(u32, __builtin_convertvector(q, bf16x2));
}
// Orders magnitudes, zero above all: a value below TINY_KEY is not zero and loses bits of its third part.
__device__ __forceinline__ u32 tiny_key(float x) { return (__float_as_uint(x) << 1) - 1u; }
constexpr u32 TINY_KEY = (u32)(27u << 24) - 1u;   // the key of 2^-100 (biased exponent 27)

// Packed layout: [group][block of 32 rows][16-row half][part][lane][8 values].  Lane (r, q) = (lane % 16, lane / 16) holds row r
// and the k-values 32 group + 8 q .. + 7.  flags[block][chunk of groups]: x bit 0 a tiny value, bit 1 a big one; y bit r row
// r is not all zero.
__global__ __launch_bounds__(256) void gemm_split_pack_kernel(const float *a, int M, int K, long long lda, int vec, int ng, int mb,
                                                               u32x4 *packed, uint2 *flags) {
    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x >> 6;
    const int r = lane & 15, q = lane >> 4;
    const int block = blockIdx.y;
    const int group = blockIdx.x * PACK_GROUPS + wave;
    u32 tiny = ~0u, rows = 0u;
    float big = 0.f;
    if (group < ng) {
        const int k = group * SG + q * 8;
#pragma unroll
        for (int f = 0; f < 2; f++) {
            const int row = block * 32 + f * 16 + r;
            const float *p = a + (long long)row * lda + k;
            f32x4 x[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
            if (row < M) {
#pragma unroll
                for (int d = 0; d < 2; d++) {
                    if (vec && k + d * 4 + 3 < K) {
                        x[d] = *reinterpret_cast<const f32x4 *>(p + d * 4);
                    } else {
#pragma unroll
                        for (int c = 0; c < 4; c++)
                            if (k + d * 4 + c < K) x[d][c] = p[d * 4 + c];
                    }
                }
            }
            u32x4 part[3];
            float most = 0.f;
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const float u = x[c >> 1][2 * (c & 1)], v = x[c >> 1][2 * (c & 1) + 1];
                u32 p1, p2, p3;
                split_pair(u, v, p1, p2, p3);
                part[0][c] = p1;
                part[1][c] = p2;
                part[2][c] = p3;
                tiny = min(tiny, min(tiny_key(u), tiny_key(v)));
                most = fmaxf(most, fmaxf(fabsf(u), fabsf(v)));
            }
            u32x4 *out = packed + (((long long)group * mb + block) * 2 + f) * 3 * WAVE + lane;
#pragma unroll
            for (int p3 = 0; p3 < 3; p3++) out[p3 * WAVE] = part[p3];
            const u64 nz = __ballot(most > 0.f);                     // (a NaN: the result tells)
            rows |= ((u32)(nz | nz >> 16 | nz >> 32 | nz >> 48) & 0xFFFFu) << (f * 16);
            big = fmaxf(big, most);
        }
    }
    __shared__ u32 seen[4][2];
    const u64 t = __ballot(tiny < TINY_KEY), b = __ballot(big >= SPLIT_BIG);
    if (lane == 0) {
        seen[wave][0] = (t ? 1u : 0u) | (b ? 2u : 0u);
        seen[wave][1] = rows;
    }
    __syncthreads();
    if (threadIdx.x == 0)
        flags[(long long)block * gridDim.x + blockIdx.x] = make_uint2(seen[0][0] | seen[1][0] | seen[2][0] | seen[3][0], seen[0][1] | seen[1][1] | seen[2][1] | seen[3][1]);
}

struct SplitArgs {
    GemmArgs g;
    const u32x4 *packed;
    const uint2 *flags;
    int ng, mb, chunks;                       // groups of k, blocks of 32 rows, flag words per block
    int gslice;                               // groups per slice of K (blockIdx.y); ng when K is not split
};

// The wave's blocks once more on the fp32 matrix cores, straight from memory (k-values k0 .. k1).
template <bool BT, int RB>
__device__ __forceinline__ void gemm_recompute(const GemmArgs &g, f32x4 (&acc)[RB][2], int m0, int n0, int r, int q, int k0, int k1) {
#pragma unroll
    for (int i = 0; i < RB; i++)
#pragma unroll
        for (int d = 0; d < 2; d++) acc[i][d] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int k = k0; k < k1; k += 4) {
        const int kk = k + q;
        const bool in = kk < k1;
        float b[2];
#pragma unroll
        for (int d = 0; d < 2; d++) {
            const int c = min(n0 + d * 16 + r, g.N - 1);
            b[d] = in ? (BT ? g.b[(long long)c * g.ldb + kk] : g.b[(long long)kk * g.ldb + c]) : 0.f;
        }
#pragma unroll
        for (int i = 0; i < RB; i++) {
            const float a = in ? g.a[(long long)min(m0 + i * 16 + r, g.M - 1) * g.lda + kk] : 0.f;
#pragma unroll
            for (int d = 0; d < 2; d++) acc[i][d] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b[d], acc[i][d], 0, 0, 0);
        }
    }
}

// Whether any of the wave's 32 weight columns holds a tiny non-zero value (bit 0) or a big one (bit 1).
template <bool BT>
__device__ __forceinline__ u32 gemm_scan_weights(const GemmArgs &g, int n0, int lane, int k0, int k1) {
    const int c = min(n0 + (lane & 31), g.N - 1);
    u32 tiny = ~0u;
    float big = 0.f;
    for (int k = k0 + (lane >> 5); k < k1; k += 2) {
        const float b = BT ? g.b[(long long)c * g.ldb + k] : g.b[(long long)k * g.ldb + c];
        tiny = min(tiny, tiny_key(b));
        big = fmaxf(big, fabsf(b));
    }
    return (__any(tiny < TINY_KEY) ? 1u : 0u) | (__any(big >= SPLIT_BIG) ? 2u : 0u);
}

// Waits until at most N of this wave's loads are in flight (direct loads into LDS count like any other; the compiler does
// not see that they are waited for here), and for its LDS reads; loads_barrier then waits for every wave of the workgroup.
template <int N>
__device__ __forceinline__ void loads_wait() {
    static_assert(N >= 0 && N < 64, "vmcnt is six bits");
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}
template <int N>
__device__ __forceinline__ void loads_barrier() {
    static_assert(N >= 0 && N < 64, "vmcnt is six bits");
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// A direct load into LDS, in assembly because the compiler, given the builtin, waits for every such load before any LDS
// read it cannot tell apart from it; "memory" keeps the LDS reads and the waits above on their side of it.  16 (4) bytes
// per lane from base + off go to LDS at lds + 16 (4) lane.
template <int BYTES>
__device__ __forceinline__ void load_to_lds(const char *base, u32 off, u32 lds) {
    if (BYTES == 16) asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory");
    else asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory");
}

// VEC: the weights' 128-bit loads are legal; else they are copied value by value (k, for [K,N] also n, clamped into the
// matrix: the packed operand is zero there, or the column is not stored).  A workgroup has NW x KH waves: NW side by
// side along N, and KH of each of those take turns along K (KH = 2: two waves share a SIMD also where a narrow tile is all a
// CU gets: one's loads, splits and waits under the other's matrix instructions).  SW: stages of weights in LDS.
// (One instance, the 256 x 256 tile over [K,N] weights value by value, has two registers in scratch; a 128 x 256 tile without them is
// slower all the same: 256 x 4096 @ 4096 x 128257 1116 us against 1235.)
template <bool BT, bool VEC, int IB, int NW, int KH, int SW, int EPI>
__global__ __launch_bounds__(64 * NW * KH) void gemm_split_kernel(SplitArgs s) {
    constexpr int AC = (IB * 6 + NW - 1) / NW;                       // 1 KiB pieces of A's groups each wave copies (some twice)
    constexpr int WC = VEC ? 4 : 16;                                 // direct loads of a wave's 4 KiB of weights per group
    constexpr int A_VEC = IB * SG_BYTES / 16;                        // 16-byte words of a group of A
    constexpr int A_STAGE = KH * A_VEC, W_STAGE = NW * KH * 256;     // .. of a step's activations, of its weights
    __shared__ __attribute__((aligned(16))) u32x4 lds[2 * A_STAGE + SW * W_STAGE];
    u32x4 *const ra = lds, *const rw = lds + 2 * A_STAGE;

    const GemmArgs &g0 = s.g;
    const int tid = threadIdx.x, lane = tid & (WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave % NW, kh = wave / NW;
    const int r = lane & 15, q = lane >> 4;
    const int mt = (g0.M + 32 * IB - 1) / (32 * IB), nt = (g0.N + 32 * NW - 1) / (32 * NW);
    int tile_m, tile_n;
    {
        const int id = blockIdx.x;
        const int full = (nt / NUM_XCD) * NUM_XCD * mt;              // ids covered by whole groups of 8 tile columns
        if (id < full) {
            const int xcd = id % NUM_XCD, x = id / NUM_XCD;
            tile_m = x % mt;
            tile_n = (x / mt) * NUM_XCD + xcd;
        } else {
            const int x = id - full;
            tile_m = x % mt;
            tile_n = (nt / NUM_XCD) * NUM_XCD + x / mt;
        }
        if (id >= mt * nt) return;
    }
    const int m0 = tile_m * 32 * IB, n0 = tile_n * 32 * NW;
    const int ncol = n0 + wn * 32;                                   // the wave's first column
    const int gfirst = (int)blockIdx.y * s.gslice;
    const int ns = min(s.gslice, s.ng - gfirst) / KH;                // this workgroup's steps of KH groups

    // A tile's stage of packed activations is contiguous.  (Where the batch ends inside the tile the copy runs on into
    // what follows, at the end of the operand into the workspace's padding: rows that are never stored.)
    const int blocks = min(IB, s.mb - tile_m * IB);
    const long long astep = (long long)s.mb * SG_BYTES;              // bytes of a group
    const char *const abase = (const char *)s.packed + (gfirst + kh) * astep + tile_m * IB * SG_BYTES + min(wn * AC, IB * 6 - AC) * 1024;
    // A wave's weights of a group, 32 columns of C x 32 k, in LDS: W[N,K] as rows of eight 16-byte words, word c of row n at
    // c ^ ((n >> 1) & 7): the operand reads of 16 consecutive rows fall into 16 different bank groups; [K,N] as rows of
    // 32 columns, row k at k ^ ((k >> 3) & 1) with its halves swapped from k = 16 on, so that the four 16-lane groups of a
    // wave, 8 k apart, read different banks.
    // Each lane's source as a byte offset from an address the wave shares, 16 bytes low to stay positive.
    const int wn0 = min(ncol, g0.N - 1);
    const char *const wbase = (const char *)(BT ? g0.b + (long long)wn0 * g0.ldb + (long long)(gfirst + kh) * SG : g0.b + wn0 + (long long)(gfirst + kh) * SG * g0.ldb) - 16;
    const long long wstep = BT ? SG * 4 : (long long)SG * g0.ldb * 4;
    auto weight_offsets = [&](u32 (&off)[WC], int last) {            // last: the last k of the group a load may start at
#pragma unroll
        for (int j = 0; j < WC; j++) {
            const int word = VEC ? j * WAVE + lane : j * 16 + (lane >> 2), e = VEC ? 0 : lane & 3;   // 16-byte word of the stage, value in it
            const int row = word >> 3, c = word & 7;
            const int n = BT ? row : (c ^ ((row >> 4) << 2)) * 4 + e, k = BT ? ((c ^ ((row >> 1) & 7)) << 2) + e : row ^ ((row >> 3) & 1);
            const int nn = min(wn0 + n, g0.N - (BT || !VEC ? 1 : 4)) - wn0, kk = min(k, last);
            off[j] = 16u + (BT ? (u32)nn * (u32)g0.ldb + (u32)kk : (u32)kk * (u32)g0.ldb + (u32)nn) * 4u;
        }
    };
    u32 woff[WC];
    weight_offsets(woff, SG);
    const u32 lds0 = (u32)(uintptr_t)(__attribute__((address_space(3))) char *)lds;
    // The XCDs walk K from different starts (and wrap): with the usual K the weights' rows are a large power of two apart, and
    // workgroups all walking in step would crowd a few memory channels (M = 64: 143 us against 158 without; every tile
    // column a start of its own: 146, but at M = 256, where the packed activations then no longer stay in an XCD's L2, 1348
    // against 1216 us).
    const int rot = (int)((unsigned)(tile_n % NUM_XCD) * (unsigned)ns / (unsigned)NUM_XCD);
    auto place = [&](int step_no) {                                  // (past the end: the last step again, not used)
        const int i = min(step_no, ns - 1) + rot;
        return (i >= ns ? i - ns : i) * KH;
    };
    // One piece of the loads of a step: A's into its stage u, the weights' into theirs.
    auto load_a = [&](const char *from, int u, int c) {
        load_to_lds<16>(from + c * 1024, lane * 16, lds0 + (u32)((u * A_STAGE + kh * A_VEC) * 16 + (min(wn * AC, IB * 6 - AC) + c) * 1024));
    };
    u32 wcur[WC];                                                    // this step's offsets, set by begin_w
    auto begin_w = [&](int i) -> const char * {
        const int last = g0.K - (VEC && BT ? 4 : 1) - (gfirst + kh + i) * SG;   // (VEC and BT: K is a multiple of 4)
        const char *from = wbase + i * wstep;
#pragma unroll
        for (int j = 0; j < WC; j++) wcur[j] = woff[j];
        if (last < (VEC && BT ? SG - 4 : SG - 1)) {                  // k clamped into the matrix: the packed operand is zero there
            const int back = last < 0 ? ((-last + SG - 1) / SG) * SG : 0;   // (a group wholly past K: an earlier one's addresses)
            weight_offsets(wcur, last + back);
            from -= BT ? (long long)back * 4 : (long long)back * g0.ldb * 4;
        }
        return from;
    };
    auto load_w = [&](const char *from, int u, int j) {
        load_to_lds<VEC ? 16 : 4>(from, wcur[j], lds0 + (u32)((2 * A_STAGE + u * W_STAGE + wave * 256) * 16 + j * (VEC ? 1024 : 256)));
    };

    constexpr int RB = 2 * IB;                                       // blocks of 16 rows
    f32x4 acc[RB][2];
#pragma unroll
    for (int i = 0; i < RB; i++)
#pragma unroll
        for (int d = 0; d < 2; d++) acc[i][d] = f32x4{0.f, 0.f, 0.f, 0.f};
    f32x4 raw[2];                                                    // eight weights of column 16 d + r, as stored
    auto read_raw = [&](int u, int d) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const u32x4 *const box = rw + u * W_STAGE + wave * 256;
            if (BT) {
                const int n = d * 16 + r;
                raw[j] = __builtin_bit_cast(f32x4, box[n * 8 + ((q * 2 + j) ^ ((n >> 1) & 7))]);
            } else {
#pragma unroll
                for (int c = 0; c < 4; c++) {                        // k = 8 q + 4 j + c
                    const int row = (q * 8 + j * 4 + c) ^ (q & 1);
                    raw[j][c] = ((const float *)box)[row * 32 + ((d ^ (q >> 1)) * 16) + r];
                }
            }
        }
    };
    u32x4 part[2][2][3];                                             // [this group, the next][d]: the weights' parts
    auto split_piece = [&](int next, int d, int c) {
        u32 p1, p2, p3;
        split_pair(raw[c >> 1][2 * (c & 1)], raw[c >> 1][2 * (c & 1) + 1], p1, p2, p3);
        part[next][d][0][c] = p1;
        part[next][d][1][c] = p2;
        part[next][d][2][c] = p3;
    };
    u32x4 fr[2][3];                                                  // A's operands of a block, read one block ahead
    auto read_frag = [&](int u, int i, u32x4 (&x)[3]) {
        const u32x4 *p = ra + u * A_STAGE + kh * A_VEC + i * 3 * WAVE + lane;
#pragma unroll
        for (int c = 0; c < 3; c++) x[c] = p[c * WAVE];
    };
    // Half f of a group's blocks: their operands are read a block ahead; `loads` issues its share of a step's loads before each
    // block; in the second half the second column
    // block of the next group's weights (raw) is split piece by piece between the matrix instructions.
    auto multiply = [&](int u, int cur, int f, auto &&loads) {
#pragma unroll
        for (int i = f * IB; i < (f + 1) * IB; i++) {
            if (i + 1 < RB) read_frag(u, i + 1, fr[(i + 1) & 1]);
            loads(i - f * IB);
            if (f == 1) {
#pragma unroll
                for (int c = (i - IB) * 4 / IB; c < (i - IB + 1) * 4 / IB; c++) split_piece(cur ^ 1, 1, c);
            }
            const bf16x8 a1 = __builtin_bit_cast(bf16x8, fr[i & 1][0]), a2 = __builtin_bit_cast(bf16x8, fr[i & 1][1]), a3 = __builtin_bit_cast(bf16x8, fr[i & 1][2]);
#pragma unroll
            for (int d = 0; d < 2; d++) {
                const bf16x8 b1 = __builtin_bit_cast(bf16x8, part[cur][d][0]), b2 = __builtin_bit_cast(bf16x8, part[cur][d][1]), b3 = __builtin_bit_cast(bf16x8, part[cur][d][2]);
                f32x4 t = acc[i][d];
                t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a3, b1, t, 0, 0, 0);
                t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b3, t, 0, 0, 0);
                t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2, b2, t, 0, 0, 0);
                t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2, b1, t, 0, 0, 0);
                t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b2, t, 0, 0, 0);
                t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b1, t, 0, 0, 0);
                acc[i][d] = t;
            }
            __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);       // the operand reads first
#pragma unroll
            for (int x = 0; x < 12; x++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // one matrix instruction ..
                __builtin_amdgcn_sched_group_barrier(0x002, IB >= 8 ? 1 : 2, 0);   // .. and what fits under it
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // Step si multiplies its KH groups out of A's stage si % 2; part[cur] holds this wave's weights' parts.  When every wave has
    // begun it, A's stage of step si - 1 is free for step si + 1; the weights' loads run SW - 1 steps ahead.  In the middle
    // of the step the wave's weights of the next step have landed and are split during its second half.  With three stages of
    // weights the loads are spread over the step, A's over its first half, theirs over the second (all at once they queue up in
    // front of the matrix instructions); with two they are needed half a step after they can be issued, and are issued at once.
    {
        const char *from = begin_w(place(0));
#pragma unroll
        for (int j = 0; j < WC; j++) load_w(from, 0, j);
        from = abase + place(0) * astep;
#pragma unroll
        for (int c = 0; c < AC; c++) load_a(from, 0, c);
        if (SW == 3) {
            from = begin_w(place(1));
#pragma unroll
            for (int j = 0; j < WC; j++) load_w(from, 1, j);
        }
    }
    loads_wait<SW == 2 ? AC : AC + WC>();
#pragma unroll
    for (int d = 0; d < 2; d++) {
        read_raw(0, d);
#pragma unroll
        for (int c = 0; c < 4; c++) split_piece(0, d, c);
    }
    static_assert(SW == 2 || SW == 3, "stages");
    int uw = SW - 1;                                                 // the weights' stage that is loaded next
    auto step = [&](int si, int cur) {                               // cur = si % 2, a constant after inlining
        loads_barrier<SW == 2 ? 0 : WC>();
        read_frag(cur, 0, fr[0]);
        const char *const fa = abase + place(si + 1) * astep, *const fw = begin_w(place(si + SW - 1));
        auto some_a = [&](int b) {
#pragma unroll
            for (int c = b * AC / IB; c < (b + 1) * AC / IB; c++) load_a(fa, cur ^ 1, c);
        };
        auto some_w = [&](int b) {
#pragma unroll
            for (int j = b * WC / IB; j < (b + 1) * WC / IB; j++) load_w(fw, uw, j);
        };
        __builtin_amdgcn_sched_barrier(0);
        if (SW == 2) {
            multiply(cur, cur, 0, [&](int b) {
                if (b == 0) {
#pragma unroll
                    for (int j = 0; j < WC; j++) load_w(fw, uw, j);
#pragma unroll
                    for (int c = 0; c < AC; c++) load_a(fa, cur ^ 1, c);
                }
            });
        } else {
            multiply(cur, cur, 0, some_a);
        }
        loads_wait<SW == 2 ? 0 : AC>();
        const int us = SW == 2 ? uw : uw == 0 ? SW - 1 : uw - 1;     // the weights' stage of step si + 1
        read_raw(us, 0);
#pragma unroll
        for (int c = 0; c < 4; c++) split_piece(cur ^ 1, 0, c);
        read_raw(us, 1);
        __builtin_amdgcn_sched_barrier(0);
        if (SW == 2) multiply(cur, cur, 1, [](int) {});
        else multiply(cur, cur, 1, some_w);
        uw = uw + 1 == SW ? 0 : uw + 1;
    };
    int si = 0;
    for (; si + 2 <= ns; si += 2) {
        step(si, 0);
        step(si + 1, 1);
    }
    if (si < ns) step(si, 0);                                        // uniform
    loads_barrier<0>();                                              // (the loads past the end)

    // The KH waves of a column share out its blocks' sums: each finishes FB of them.
    constexpr int FB = RB / KH;
    f32x4 fin[FB][2];
    if constexpr (KH == 1) {
#pragma unroll
        for (int i = 0; i < FB; i++)
#pragma unroll
            for (int d = 0; d < 2; d++) fin[i][d] = acc[i][d];
    } else {
        f32x4 *const box = reinterpret_cast<f32x4 *>(lds) + lane;   // [wave][block][d][lane]
        static_assert(KH == 2 && NW * KH * FB * 2 * WAVE <= 2 * A_STAGE + SW * W_STAGE, "hand-over");
#pragma unroll
        for (int i = 0; i < FB; i++)
#pragma unroll
            for (int d = 0; d < 2; d++) box[((wave * FB + i) * 2 + d) * WAVE] = kh ? acc[i][d] : acc[FB + i][d];
        lds_barrier();
        const int other = wave ^ NW;
#pragma unroll
        for (int i = 0; i < FB; i++)
#pragma unroll
            for (int d = 0; d < 2; d++) fin[i][d] = (kh ? acc[FB + i][d] : acc[i][d]) + box[((other * FB + i) * 2 + d) * WAVE];
        if (EPI == 2) lds_barrier();                                 // (the epilogue stages there)
    }
    const int mfin = m0 + kh * FB * 16;                              // the first of this wave's rows

    // Operands the parts cannot hold?
    u32 aflags = 0u, live[FB / 2];                                   // live[i]: the rows of 32-row block i that are not all zero
#pragma unroll
    for (int i = 0; i < FB / 2; i++) live[i] = 0u;
#pragma unroll
    for (int i = 0; i < FB / 2; i++)
        for (int c = lane; c < s.chunks && kh * (FB / 2) + i < blocks; c += WAVE) {
            const uint2 f = s.flags[((long long)tile_m * IB + kh * (FB / 2) + i) * s.chunks + c];
            aflags |= f.x;
            live[i] |= f.y;
        }
#pragma unroll
    for (int o = 1; o < WAVE; o <<= 1) {
        aflags |= (u32)__shfl_xor((int)aflags, o, WAVE);
#pragma unroll
        for (int i = 0; i < FB / 2; i++) live[i] |= (u32)__shfl_xor((int)live[i], o, WAVE);
    }
    float poison = 0.f, least = INFINITY;
#pragma unroll
    for (int i = 0; i < FB; i++)
#pragma unroll
        for (int d = 0; d < 2; d++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int row = i * 16 + q * 4 + v;
                if (mfin + row < g0.M) poison += fin[i][d][v] * 0.f;
                if (((live[i / 2] >> (row & 31)) & 1u) && ncol + d * 16 + r < g0.N) least = fminf(least, fabsf(fin[i][d][v]));
            }
    const int k0 = gfirst * SG, k1 = min((gfirst + ns * KH) * SG, g0.K);
    bool again = __any(poison != poison);
    if (!again && (aflags || __any(least < SPLIT_SMALL_RESULT))) {
        const u32 wflags = gemm_scan_weights<BT>(g0, ncol, lane, k0, k1);
        again = ((aflags & 1u) && (wflags & 2u)) || ((aflags & 2u) && (wflags & 1u)) || (((aflags | wflags) & 1u) && __any(least < SPLIT_SMALL_RESULT));
    }
    GemmArgs g = s.g;
    if (again) gemm_recompute<BT, FB>(g, fin, mfin, ncol, r, q, k0, k1);
    if (s.gslice < s.ng) {                                           // a slice of K: the partial product, without bias
        g.c = g.ws + (long long)blockIdx.y * g.M * g.N;
        g.ldc = g.N;
        g.bias = nullptr;
    }
    static_assert(gemm_stage_bytes(NW * KH) <= (2 * A_STAGE + SW * W_STAGE) * 16, "the epilogue's stage");
    gemm_finish<EPI, 16, NW * KH>(g, fin, mfin, ncol, lds);
}

template <int IB, int NW, int KH, int SW, int EPI>
static void launch_split(const SplitArgs &s, bool bt, bool vec, hipStream_t st) {
    const long long mt = (s.g.M + 32 * IB - 1) / (32 * IB), nt = (s.g.N + 32 * NW - 1) / (32 * NW);
    const dim3 gr((unsigned)(mt * nt), (unsigned)((s.ng + s.gslice - 1) / s.gslice)), bl(64 * NW * KH);
    if (bt) {
        if (vec) hipLaunchKernelGGL((gemm_split_kernel<true, true, IB, NW, KH, SW, EPI>), gr, bl, 0, st, s);
        else hipLaunchKernelGGL((gemm_split_kernel<true, false, IB, NW, KH, SW, EPI>), gr, bl, 0, st, s);
    } else if constexpr (EPI == 0) {
        if (vec) hipLaunchKernelGGL((gemm_split_kernel<false, true, IB, NW, KH, SW, EPI>), gr, bl, 0, st, s);
        else hipLaunchKernelGGL((gemm_split_kernel<false, false, IB, NW, KH, SW, EPI>), gr, bl, 0, st, s);
    }
}
template <int EPI>
static void launch_split_tile(const SplitArgs &s, int tile, bool bt, bool vec, hipStream_t st) {
    if (tile == 0) launch_split<2, 4, 2, 3, EPI>(s, bt, vec, st);
    else if (tile == 1) launch_split<4, 4, 2, 2, EPI>(s, bt, vec, st);
    else if (tile == 2) launch_split<4, 8, 1, 3, EPI>(s, bt, vec, st);
    else launch_split<8, 8, 1, 2, EPI>(s, bt, vec, st);
}

hipError_t launch_gemm_split(const GemmArgs &g, bool bt, int tile, void *workspace, hipStream_t st) {
    SplitArgs s;
    s.g = g;
    s.ng = (g.K + 2 * SG - 1) / (2 * SG) * 2;                        // (pairs of groups: padded with zeros)
    s.mb = (g.M + 31) / 32;
    s.chunks = (s.ng + PACK_GROUPS - 1) / PACK_GROUPS;
    s.packed = reinterpret_cast<const u32x4 *>(workspace);
    uint2 *flags = reinterpret_cast<uint2 *>((char *)workspace + (size_t)s.ng * s.mb * SG_BYTES + 8 * SG_BYTES);
    s.flags = flags;
    s.gslice = g.ksplit > 1 ? g.kslice / SG : s.ng;                  // (even)
    hipLaunchKernelGGL(gemm_split_pack_kernel, dim3((unsigned)s.chunks, (unsigned)s.mb), dim3(256), 0, st, g.a, g.M, g.K, g.lda,
                       g.vec_a ? 1 : 0, s.ng, s.mb, reinterpret_cast<u32x4 *>(workspace), flags);
    const bool vec = g.vec_b && (bt ? g.K : g.N) % 4 == 0;
    if (g.ksplit > 1) launch_split_tile<0>(s, tile, bt, vec, st);
    else if (g.cand) launch_split_tile<2>(s, tile, bt, vec, st);
    else if (g.best) launch_split_tile<1>(s, tile, bt, vec, st);
    else launch_split_tile<0>(s, tile, bt, vec, st);
    return hipGetLastError();
}

}  // namespace born
