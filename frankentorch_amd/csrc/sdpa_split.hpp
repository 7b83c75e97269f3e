// Attention over many queries on the bf16 matrix units (csrc/sdpa_split.hip), used by csrc/sdpa.hip.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "ft_kernel_hip.h"

namespace fth {

// True when the kernel covers the problem and is the faster one: no mask, 0 < scale <= 2^20, d_k == d_v in {64, 128}, K and V row
// strides that are not negative. Operands are 16-byte aligned with strides that are multiples of four (the caller checks).
bool sdpa_split_pays(const fth_sdpa_desc &d, float scale);
int32_t sdpa_split_f32(const fth_sdpa_desc &d, float scale, const float *q, const float *k, const float *v, float *out, hipStream_t st);

}  // namespace fth
