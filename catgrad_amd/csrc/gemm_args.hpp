// Kernel arguments of the batched matrix products (matmul.hip, split_gemm.hip).
#pragma once

#include "common.hpp"
#include "device_utils.hpp"
#include "narrow_route.hpp"

namespace cg {

struct MmArgs {
    const uint32_t *A;
    const uint32_t *B;
    uint32_t *C;
    uint32_t M, N, K;
    int64_t a_sm, a_sk, b_sk, b_sn;
    uint32_t nb;                    // collapsed batch axes
    uint32_t bd[kMaxBatchAxes];     // extents, innermost first
    FastDiv bdiv[kMaxBatchAxes];
    int64_t a_bs[kMaxBatchAxes], b_bs[kMaxBatchAxes];
    uint32_t batch;
    uint32_t a_vec, b_vec;          // 16-byte loads along the unit-stride axis are legal
    uint32_t ksplit;                // tiled kernels: values of k per workgroup along grid.z (a multiple of 32), 0 = all of K
    uint32_t n_tiles;               // mfma_gemm_dlds_kernel: columns of tiles that it computes, from the first; 0 = all
    uint32_t c_fmt;                 // mfma_gemm_dlds_kernel: kFmtWords, or the operands' narrow format: C holds its patterns, rounded in the store
};

__device__ __forceinline__ void batch_offsets(const MmArgs &a, uint32_t b, int64_t &oa, int64_t &ob) {
    oa = 0;
    ob = 0;
    for (uint32_t d = 0; d < a.nb; d++) {
        uint32_t q = fastdiv(b, a.bdiv[d]);
        int64_t i = (int64_t)(b - q * a.bd[d]);
        b = q;
        oa += i * a.a_bs[d];
        ob += i * a.b_bs[d];
    }
}

// The f32 products of more than eight rows (split_gemm.hip).  `a` complete but for ksplit; C is the row-major result.
// a_mfast / b_nfast: the operand's rows, not k, are its unit-stride axis.
int launch_split_gemm(cg_backend *be, MmArgs a, bool a_mfast, bool b_nfast);
// The same for a few dozen rows whose operands have k contiguous in 16-byte pieces (split_thin.hip), 16 `high` rows per workgroup, and
// what that takes in microseconds.
double thin_gemm_cost(const cg_backend *be, const MmArgs &a, int *high);
int launch_thin_gemm(cg_backend *be, const MmArgs &a, int high);


// y[rows, n] = x[rows, k] . w[n, k]^T of patterns of one narrow format (block_products.hip); pitches in elements; y's rows y_pitch
// apart (0: dense), words or patterns of that format.  kDeclined: operands that fits_narrow_tiles does not take or that are not 16-byte aligned.
int launch_narrow_tiles(cg_backend *be, int fmt, const void *x, int64_t x_pitch, int64_t rows, const void *w, int64_t w_pitch, int64_t n, int64_t k, void *y, int y_fmt,
                        int64_t y_pitch = 0);

} // namespace cg
