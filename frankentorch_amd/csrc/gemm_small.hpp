// fp32 products of few rows, or of little work: one launch, K split over the wavefronts of a workgroup (gemm_small.hip).
#pragma once

#include "common.hpp"

namespace fth {

// C = alpha * A . B^T (trans_b: B is [n, k]) or A . B (B is [k, n]), then bias, GELU, residual; `batch` of them, stride_* apart.
struct SmallGemm {
    const float *a, *b;
    float *c;
    const float *bias, *residual;
    int64_t m, n, k, lda, ldb, ldc, stride_a, stride_b, stride_c, batch;
    float alpha;
    int epilogue;
    bool trans_b;
};

// Runs the product when this is the kernel for it (rows of A, and of a [n, k] B, are 16-byte aligned: the caller checks);
// false, with nothing launched, otherwise.
bool small_gemm(const SmallGemm &g, hipStream_t st, int32_t *rc);

}  // namespace fth
