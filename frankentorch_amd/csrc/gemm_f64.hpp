// float64 products that leave the large-tile kernels short of work (gemm_f64.hip).
#pragma once

#include "common.hpp"

namespace fth {

// C = alpha * op(A) . op(B), then bias, GELU, residual; A is [m, k] or, trans_a, [k, m]; B is [k, n] or, trans_b, [n, k].
struct SmallGemm64 {
    const double *a, *b;
    double *c;
    const double *bias, *residual;
    int64_t m, n, k, lda, ldb, ldc, stride_a, stride_b, stride_c, batch;
    double alpha;
    int epilogue;
    bool trans_a, trans_b;
};

// Runs the product when this is the kernel for it; false, with nothing launched, otherwise.
bool small_gemm_f64(const SmallGemm64 &g, hipStream_t st, int32_t *rc);

}  // namespace fth
