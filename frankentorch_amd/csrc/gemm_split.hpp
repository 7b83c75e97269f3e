// fp32 products on the bf16 matrix units: exact three-way split of both operands (gemm_split.hip).
#pragma once

#include "common.hpp"

namespace fth {

// C = alpha * A . B^T (+ bias, GELU, residual). Element (row, k) of an operand is ptr[row * row_stride + k * k_stride], one of
// the strides being 1; rows of A are rows of C, rows of B are columns of C.
struct SplitGemm {
    const float *a, *b;
    int64_t a_rs, a_ks, b_rs, b_ks;
    float *c;
    const float *bias, *residual;
    float *rowmax;  // as GemmArgs::rowmax, or NULL
    int64_t m, n, k, ldc;
    float alpha;
    int epilogue;
};

// How the fp32 kernel that the split product would stand in for reads its operands.
enum class SplitRival { Direct, Copied, Vector, Single };  // straight into LDS, so after a transposed copy of A, in 128-bit loads, element by element

// True when the split product is the faster one for this shape and its planes fit the scratch bound.
bool split_gemm_pays(const SplitGemm &g, SplitRival rival);
// Runs it. Returns false, with nothing launched, when the scratch memory cannot be had.
bool split_gemm(const SplitGemm &g, hipStream_t st, int32_t *rc);

}  // namespace fth
