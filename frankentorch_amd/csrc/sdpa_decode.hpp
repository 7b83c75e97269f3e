// Few-query attention against a long K/V cache (csrc/sdpa_decode.hip), used by csrc/sdpa.hip.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "ft_kernel_hip.h"

namespace fth {

// True when the key-split kernel covers the problem: seq_q <= 8, no causal flag, d_k == d_v in {32, 64, 128}. Operands are
// 16-byte aligned with strides that are multiples of four (the caller checks). short_alternative: the key-split kernel for small
// problems would take the call.
bool sdpa_decode_applies(const fth_sdpa_desc &d, bool short_alternative);
// Runs it. Returns false, with nothing launched, when the scratch memory cannot be had.
bool sdpa_decode_f32(const fth_sdpa_desc &d, float scale, const float *q, const float *k, const float *v, const float *mask,
                     int64_t mask_bh_stride, float *out, bool short_alternative, hipStream_t st, int32_t *rc);

}  // namespace fth
