// The exact split of floats into three bf16 parts, and the vector types that its users share.
//
// A float has 24 significant bits; three bf16 values hold 8 each. Rounding to nearest three times, x = x0 + x1 + x2 EXACTLY
// (x0 = bf16(x), x1 = bf16(x - x0), x2 = x - x0 - x1, which has at most 8 significant bits left). A product of two such sums is
// formed from six products of parts, x0 y0, x0 y1, x1 y0, x1 y1, x0 y2, x2 y0; the three left out are below 2^-24 |x y| together
// and of either sign.
#pragma once

#include <cstdint>

namespace fth {

using bf16x8 = __attribute__((ext_vector_type(8))) __bf16;
using bf16x2 = __attribute__((ext_vector_type(2))) __bf16;
using f32x2 = __attribute__((ext_vector_type(2))) float;
using f32x4 = __attribute__((ext_vector_type(4))) float;
using f32x16 = __attribute__((ext_vector_type(16))) float;
using u32x4 = __attribute__((ext_vector_type(4))) uint32_t;

constexpr int kPlanes = 3;

__device__ __forceinline__ uint32_t pack_bf16(float x, float y) {
    const f32x2 v = {x, y};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));  // v_cvt_pk_bf16_f32: to nearest even
}
__device__ __forceinline__ float lo_f32(uint32_t p) { return __builtin_bit_cast(float, p << 16); }
__device__ __forceinline__ float hi_f32(uint32_t p) { return __builtin_bit_cast(float, p & 0xffff0000u); }

// The three parts of two floats, one dword each.
__device__ __forceinline__ void split2(float x, float y, uint32_t &p0, uint32_t &p1, uint32_t &p2) {
    p0 = pack_bf16(x, y);
    x -= lo_f32(p0);
    y -= hi_f32(p0);
    p1 = pack_bf16(x, y);
    x -= lo_f32(p1);
    y -= hi_f32(p1);
    p2 = pack_bf16(x, y);
}

// The three parts of eight floats, an MFMA operand each.
__device__ __forceinline__ void split8(const float (&v)[8], u32x4 (&w)[kPlanes]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        uint32_t p0, p1, p2;
        split2(v[2 * e], v[2 * e + 1], p0, p1, p2);
        w[0][e] = p0;
        w[1][e] = p1;
        w[2][e] = p2;
    }
}

}  // namespace fth
