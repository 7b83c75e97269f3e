// Attention of 32 query rows on one wavefront with fp32 MFMAs, straight from memory: what the kernel on the bf16 matrix units
// (sdpa_split.hip) falls back to for operands that its parts cannot stand for.
#pragma once

#include <hip/hip_runtime.h>

#include "devmath.hpp"
#include "ft_kernel_hip.h"
#include "split_bf16.hpp"

namespace fth {

// Online softmax of queries q0 .. q0 + 31 over keys 0 .. 32 num_kt - 1, with the scheme of sdpa_small_kernel (sdpa.hip). Lane l holds query q0 + l % 32; o[e][r] is its output element e + D / 32 (8 (r / 4) + 4 (l / 32) + r % 4), not yet
// divided by l_run. Few registers instead of requests ahead of their use: the caller holds many, and this is rare.
template <int D>
__device__ __forceinline__ void sdpa_rows_f32(const fth_sdpa_desc &d, const float *Q, const float *K, const float *V, float c2, int q0,
                                              int num_kt, f32x16 (&o)[D / 32], float &l_run) {
    constexpr int NDT = D / 32;
    using V4 = float __attribute__((ext_vector_type(NDT)));
    const int lane = threadIdx.x & 63, lq = lane & 31, half = lane >> 5;
    const int seq_k = (int)d.seq_k, qi = q0 + lq;
    const float *qp = Q + (int64_t)(qi < (int)d.seq_q ? qi : (int)d.seq_q - 1) * d.q_row_stride + 4 * half;
#pragma unroll
    for (int e = 0; e < NDT; ++e)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[e][r] = 0.f;
    float m_run = -__builtin_inff();
    l_run = 0.f;
    for (int kt = 0; kt < num_kt; ++kt) {
        const int key0 = kt * 32;
        int krow = key0 + lq;
        krow = krow < seq_k ? krow : seq_k - 1;  // rows past the end repeat the last one; their scores are hidden
        const float *kp = K + (int64_t)krow * d.k_row_stride + 4 * half;
        f32x16 s;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
        for (int t = 0; t < D / 8; ++t) {
            const f32x4 kv = *reinterpret_cast<const f32x4 *>(kp + 8 * t), qv = *reinterpret_cast<const f32x4 *>(qp + 8 * t);
#pragma unroll
            for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[e], qv[e], s, 0, 0, 0);
            if (t % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
        float mt = -__builtin_inff();
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int key = key0 + 8 * (r >> 2) + 4 * half + (r & 3);
            const bool hidden = (d.causal && key > qi) | (key >= seq_k);
            s[r] = hidden ? -__builtin_inff() : s[r];
            mt = fmaxf(mt, s[r]);
        }
        float mlo, mhi;
        both_halves(mt, mlo, mhi);
        const float m_new = fmaxf(m_run, fmaxf(mlo, mhi));  // (a raw score)
        const float m_ref = m_new == -__builtin_inff() ? 0.f : m_new;  // nothing seen yet: the state stays empty
        const float alpha = __builtin_amdgcn_exp2f((m_run - m_ref) * c2);
        if (__any(alpha != 1.0f)) {
#pragma unroll
            for (int e = 0; e < NDT; ++e)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[e][r] *= alpha;
        }
        float psum = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float w = __builtin_amdgcn_exp2f((s[r] - m_ref) * c2);
            psum += w;
            int vrow = key0 + 8 * (r >> 2) + (r & 3) + 4 * half;
            vrow = vrow < seq_k ? vrow : seq_k - 1;
            const V4 v = *reinterpret_cast<const V4 *>(V + (int64_t)vrow * d.v_row_stride + NDT * lq);
#pragma unroll
            for (int e = 0; e < NDT; ++e) o[e] = __builtin_amdgcn_mfma_f32_32x32x2f32(v[e], w, o[e], 0, 0, 0);
            if (r % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
        float plo, phi;
        both_halves(psum, plo, phi);
        l_run = l_run * alpha + (plo + phi);
        m_run = m_new;
    }
}

}  // namespace fth
