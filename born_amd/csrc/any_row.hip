// A batch whose rows bring settings of their own, rows of any kind in one launch: a workgroup of 1024 threads per row runs the
// single-pass body (topk_row_impl.h), the three-sweep body (nucleus_row_impl.h) or the general kernel's.
//
// Up to a row per CU.  As two launches, one for the rows with a small top-k and one for the others, each leaves the CUs of the
// other's rows idle and a step takes the sum of the slowest row of either; in one it takes the larger.  In one launch, us, half
// of the rows with a top-k of up to 100 (two launches, with the three-sweep body of then, and one, with it and now): 96 x 100 003 72.6 51.3 40.4, 8 x 32 000 41.0 26.2 22.9, 32 x 128 256
// 80.5 58.7 46.8, 128 x 50 000 52.3 35.7 28.2.  Bound by the slowest row's three sweeps on one CU.  (Registers are spilled in the general kernel's body,
// as in nucleus_or_general_rows_kernel: the others take what they take alone.)  More rows than CUs keep the kernels of their own:
// a CU holds one workgroup of this one, two of theirs.  Occurrence tables too: an instance with them would double the code.
#include "nucleus_row_impl.h"
#include "topk_tail.h"

#define BORN_WIDE_BLOCK 1024
#define BORN_WIDE_NS wide_in_any
#define BORN_WIDE_BODY_ONLY
#include "sample_wide_impl.h"
#undef BORN_WIDE_BODY_ONLY
#undef BORN_WIDE_BLOCK
#undef BORN_WIDE_NS

namespace born {

#define BORN_ROW_BLOCK 1024
#define BORN_ROW_BODY_ONLY
#include "topk_row_impl.h"
#undef BORN_ROW_BODY_ONLY
#undef BORN_ROW_BLOCK

template <int MODE>
__global__ __launch_bounds__(1024) void any_row_kernel(SampleArgs a, RowConfigs rc) {
    extern __shared__ __align__(16) u64 any_dyn[];                   // (the bodies' storage, each from its start)
    __shared__ BlockScratch wide_scr;
    __shared__ int wide_int[8];
    __shared__ u64 wide_u64[4];
    const int row = (int)blockIdx.x;
    RowValues v;
    bool invalid;
    if (row_config_values(a, rc, row, ROUTE_NUCLEUS, v, invalid)) {  // workgroup-uniform, before any barrier
        if (invalid) row_config_reject(a, row);
        else nucleus_row_body<1024, false, true, true>(a, v.T, v.top_p, v.rep, v.dcut, v.freq, v.pres, nuc_reciprocal(v.T));
        return;
    }
    if (row_config(a, rc, row, ROUTE_TOPK, invalid)) {
        if (invalid) row_config_reject(a, row);
        else (topk_row_body<MODE, false, 1>)(a);
        return;
    }
    if (!row_config(a, rc, row, ROUTE_GENERAL, invalid)) return;
    if (invalid) row_config_reject(a, row);
    else wide_in_any::wide_row<false>(a, row, (lds_u64 *)any_dyn, (BORN_LDS BlockScratch *)&wide_scr, (lds_int *)wide_int, (lds_u64 *)wide_u64);
}

// (rows with a small top-k are among them: at most ROW_MAX_VOCAB logits)
static size_t any_row_lds(int V) {
    return std::max(row_pool_bytes<1>(), std::max(nucleus_lds_bytes(V), wide_lds_bytes(V)));
}

bool any_row_takes(const SampleArgs &a) { return !a.hist_counts && !a.local_counts && a.B <= device_cu_count(); }

hipError_t launch_any_rows(const SampleArgs &args, hipStream_t st, const RowConfigs &rows) {
    SampleArgs a = args;
    a.row_blocks = row_blocks(args);
    const dim3 gr((unsigned)a.B), bl(1024);
    const size_t lds = any_row_lds(a.V);
    if (rows_aligned(a.logits, a.row_stride)) hipLaunchKernelGGL(any_row_kernel<ROW_ALIGNED>, gr, bl, lds, st, a, rows);
    else if (a.V >= ROW_LOADS4_FROM) hipLaunchKernelGGL(any_row_kernel<ROW_ANY>, gr, bl, lds, st, a, rows);
    else hipLaunchKernelGGL(any_row_kernel<ROW_SHORT>, gr, bl, lds, st, a, rows);
    return hipGetLastError();
}

hipError_t configure_any_row() {
    for (const void *k : {reinterpret_cast<const void *>(any_row_kernel<ROW_ALIGNED>), reinterpret_cast<const void *>(any_row_kernel<ROW_ANY>),
                          reinterpret_cast<const void *>(any_row_kernel<ROW_SHORT>)}) {
        const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)any_row_lds(ROW_MAX_VOCAB));
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace born
