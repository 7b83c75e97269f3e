// Fused scaled-dot-product attention forward, fp32, on the bf16 matrix units.
//
// The same mathematics as sdpa_mfma_kernel (sdpa.hip): S^T = K . Q^T, online softmax, O^T = V^T . P^T; but Q, K, V and the weights P
// are each split into three bf16 parts that sum to the float exactly (split_bf16.hpp) and every product is formed from six
// products of parts with fp32 sums. Six 32 x 32 x 16 bf16 MFMAs cost 192 cycles where the eight fp32 MFMAs of the same 16 k
// cost 512.
//
// Nothing is laid out beforehand: a workgroup reads K and V as floats, splits each tile once and shares the parts through LDS. At
// 256 queries a workgroup that is 5.5 vector instructions an element of P, against 10 bytes of memory traffic an element of K and V
// for a pass of its own, and it needs no scratch memory. Unlike fp32 MFMAs, bf16 ones leave the vector unit its issue cycles: up to
// seven vector instructions of any kind used here hide behind one MFMA of 32 cycles (the dot-product instructions do not).
//
// Bound by the matrix units and the power they draw: causal, 4 x 32 heads of 2048 tokens, head size 128, 1050 -> 680 us; not causal
// 1936 -> 1235 us, 223 TFLOP/s of attention, 1.34 PFLOP/s of bf16 products. 96 heads of 1024 tokens, head size 64, 119 -> 82 us.
// Relative 2-norm error against 64 bits, fp32 MFMA kernel / here: causal 4.5e-7 / 3.0e-7, not causal 8.9e-7 / 7.1e-7 (2048 tokens);
// values of one sign 6.7e-7 / 4.4e-7, half of them zero 4.8e-7 / 4.5e-7, scores of standard deviation 8 1.8e-6 / 6.8e-7.
//
// What the parts cannot stand for: infinities, NaN, operands of 2^53 and more in Q or K (whose sums could overflow where fp32
// sums do not), values of V under 2^-110 (whose third part lies below the bf16 subnormals) where the output is small as well, and
// weights under 2^-110 where nothing else makes up the output. What a weight loses is below 2^-134 (it is 2^-126 or zero at the
// least, and the largest of a row at least one), so an output is off by at most seq_k 2^-134 max |V|: nothing that counts where it is
// 2^-96 max |V| or more. A smaller one that is not zero needs keys of large weight whose values are zero or next to it. (The largest
// |V| is kept beside the smallest for this: 0.3 us a block, 14.0 -> 14.3 us for 64 heads of 130 tokens, 681 -> 685 for the causal problem above, timed in turn.)
// A wavefront that finds a NaN, an infinity or such an output in its results, or is told of such operands, computes its 32 queries
// again with fp32 MFMAs (sdpa_rows.hpp). Tiny values in Q and K need nothing: with the partners below 2^53 and a scale of at most
// 2^20 what is lost of a score is below 2^-50.
//
// replaces sdpa_forward_f32 (crates/ft-kernel-cpu/src/lib.rs:4572-4651, 5200-5284) for problems of many queries.

#include <cfloat>
#include <cstdlib>
#include <type_traits>

#include "common.hpp"
#include "sdpa_rows.hpp"
#include "sdpa_split.hpp"
#include "split_bf16.hpp"

namespace {

using fth::bf16x8;
using fth::f32x4;
using Acc16 = fth::f32x16;
using fth::kPlanes;
using fth::u32x4;

constexpr int kXcds = 8;
constexpr float kLarge = 0x1p53f, kTinyOut = 0x1p-100f, kTinyShare = 0x1p-96f;
constexpr uint32_t kTinyBits = 0x08800000u;  // 2^-110
constexpr float kLazy = 6.0f;                // log2 units by which a score may exceed the reference m before it moves

struct SplitSdpaArgs {
    const float *q, *k, *v;
    float *out;
    fth_sdpa_desc d;
    float scale;
    int q_blocks;
    int64_t group;  // query heads per K/V head
};

__device__ __forceinline__ float nan_max(float a, float b) { return __builtin_elementwise_maximum(a, b); }
__device__ __forceinline__ bf16x8 as_bf16(u32x4 w) { return __builtin_bit_cast(bf16x8, w); }
__device__ __forceinline__ Acc16 mfma(bf16x8 a, bf16x8 b, Acc16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }

// Largest x of a wavefront (no NaN), in every lane: along rows of 16 lanes, then across them.
__device__ __forceinline__ float wave_max(float x) {
    auto step = [&](auto ctrl) __attribute__((always_inline)) {
        const int y = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), decltype(ctrl)::value, 0xf, 0xf, false);
        x = __builtin_fmaxf(x, __builtin_bit_cast(float, y));
    };
    step(std::integral_constant<int, 0x128>{});  // row_ror by 8, 4, 2, 1
    step(std::integral_constant<int, 0x124>{});
    step(std::integral_constant<int, 0x122>{});
    step(std::integral_constant<int, 0x121>{});
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, x), __builtin_bit_cast(unsigned, x), false, false);
    x = __builtin_fmaxf(__builtin_bit_cast(float, r[0]), __builtin_bit_cast(float, r[1]));
    float lo, hi;
    fth::both_halves(x, lo, hi);
    return __builtin_fmaxf(lo, hi);
}

// QW wavefronts of 32 queries each times KW wavefronts along the keys; a stage of LDS holds KEYS keys, of which a wavefront takes SUB
// sub-tiles of 32.
//   S^T[key, query]: A = K parts from LDS (lane: key l % 32, eight d from 8 (l / 32) on), B = the wavefront's Q parts in registers.
//   A lane then holds, for one query, the keys 8 (r / 4) + 4 (l / 32) + r % 4. O^T[d, query]: B = the lane's own P parts, eight
//   consecutive r an MFMA; A = V parts from LDS in the same key order, so P never leaves its lane.
// LDS, in 16-byte chunks of eight bf16: K [part][d / 8][key ^ x(d / 8)], V [part][sub, r / 8, l / 32][d]. A chunk of K is written
// by the thread that read 32 consecutive bytes of a row, and x (d / 8, twice that for rows of 64) spreads the 16 or 8 threads of a row
// over the banks; reads run over consecutive keys or d.
// A thread splits one chunk of K and one of V a stage.
// The leading product of a score follows the lower ones, so that these do not each round the full sum.
template <int D, int QW, int KW>
__global__ __launch_bounds__(64 * QW *KW, 2) void sdpa_split_kernel(const SplitSdpaArgs p) {
    constexpr int NW = QW * KW, NTH = 64 * NW;
    constexpr int KEYS = 4096 / D;                    // keys of a stage
    constexpr int SUBS = KEYS / 32, SUB = SUBS / KW;  // 32-key sub-tiles of a stage, and of a wavefront
    constexpr int PART = KEYS * D * 2;                // bytes of one part of K or V of a stage
    constexpr int STAGE = 2 * kPlanes * PART;
    constexpr int VOFF = kPlanes * PART;
    constexpr int NDT = D / 32, KSTEPS = D / 16;
    constexpr int XS = D == 128 ? 0 : 1;  // x(c) = c << XS
    static_assert(SUB >= 1 && NTH == 512, "a thread splits one chunk of K and one of V a stage");
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    __shared__ int flags[2];  // operands of 2^53 and more, tiny values of V
    __shared__ float largest[NW];  // |V| that each wavefront has split

    const fth_sdpa_desc &d = p.d;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lq = lane & 31, half = lane >> 5;
    const int qw = wave % QW, kw = wave / QW;

    // Blocks are issued longest first across all heads; a K/V head, with every query head that reads it, stays on one XCD.
    int64_t bh;
    int unit;
    {
        const int64_t pid = blockIdx.x, g = p.group, kv_heads = d.num_bh / g;
        if (kv_heads % kXcds == 0) {
            const int64_t xcd = pid % kXcds, per = d.num_bh / kXcds, w = pid / kXcds;
            unit = (int)(w / per);
            const int64_t idx = w % per;
            bh = ((idx / g) * kXcds + xcd) * g + idx % g;
        } else {
            unit = (int)(pid / d.num_bh);
            bh = pid % d.num_bh;
        }
    }
    const int64_t b = bh / d.heads, h = bh % d.heads, hk = h / p.group;
    const float *Q = p.q + b * d.q_batch_stride + h * d.q_head_stride;
    const float *K = p.k + b * d.k_batch_stride + hk * d.k_head_stride;
    const float *V = p.v + b * d.v_batch_stride + hk * d.v_head_stride;
    float *O = p.out + b * d.o_batch_stride + h * d.o_head_stride;
    const float c2 = p.scale * 1.44269502162933349609375f;  // scale * log2(e)

    const int qb = p.q_blocks - 1 - unit;
    const int q_blk0 = qb * 32 * QW, q_wave0 = q_blk0 + qw * 32, qi = q_wave0 + lq;
    const int seq_q = (int)d.seq_q, seq_k = (int)d.seq_k;
    const bool q_live = qi < seq_q;
    const int blk_last_q = q_blk0 + 32 * QW - 1 < seq_q - 1 ? q_blk0 + 32 * QW - 1 : seq_q - 1;
    const int wave_last_q = q_wave0 + 31 < seq_q - 1 ? q_wave0 + 31 : seq_q - 1;
    const int k_end = d.causal && blk_last_q + 1 < seq_k ? blk_last_q + 1 : seq_k;
    const int num_kt = (k_end + KEYS - 1) / KEYS;

    // ---- Q parts: lane holds Q[qi][16 s + 8 half + 0 .. 7] ----
    bf16x8 q0[KSTEPS], q1[KSTEPS], q2[KSTEPS];
    float q_max = 0.f;
    const float *qrow = Q + (int64_t)(q_live ? qi : seq_q - 1) * d.q_row_stride + 8 * half;  // (rows past the end repeat the last one)
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) {
        const f32x4 lo = *reinterpret_cast<const f32x4 *>(qrow + 16 * s), hi = *reinterpret_cast<const f32x4 *>(qrow + 16 * s + 4);
        float x[8];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            x[e] = lo[e];
            x[4 + e] = hi[e];
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) q_max = __builtin_fmaxf(q_max, __builtin_fabsf(x[e]));
        u32x4 w[kPlanes];
        fth::split8(x, w);
        q0[s] = as_bf16(w[0]);
        q1[s] = as_bf16(w[1]);
        q2[s] = as_bf16(w[2]);
        asm volatile("" : "+v"(q0[s]), "+v"(q1[s]), "+v"(q2[s]));  // split here, not beside everything that the loop holds
    }

    const bool q_large = __builtin_amdgcn_ballot_w64(!(q_max < kLarge)) != 0;

    // ---- loader ----
    constexpr int RL = D / 8;                       // lanes along a row of K
    constexpr int KROWS = 64 / RL, VW = D / 64;     // K rows a wavefront reads at once; wavefronts along a row of V
    f32x4 kreg[2];
    float vreg[8];
    float k_max = 0.f, v_max = 0.f;
    uint32_t v_min = 0xffffffffu;
    // Offsets that depend on the lane are worked out where they are used: registers are what this kernel is short of.
    auto my_lane = [&]() __attribute__((always_inline)) {
        int l = lane;
        asm volatile("" : "+v"(l));
        return l;
    };
    auto load_k = [&](int kt) __attribute__((always_inline)) {
        const char *kb = reinterpret_cast<const char *>(K + (int64_t)kt * KEYS * d.k_row_stride);
        const int l = my_lane(), last = seq_k - 1 - kt * KEYS;
        int row = wave * KROWS + l / RL;
        row = row < last ? row : last;  // rows past the end repeat the last one; their scores are hidden
        const uint32_t off = (uint32_t)row * ((uint32_t)d.k_row_stride * 4u) + (uint32_t)(l % RL) * 32u;
        kreg[0] = *reinterpret_cast<const f32x4 *>(kb + off);
        kreg[1] = *reinterpret_cast<const f32x4 *>(kb + off + 16);
    };
    auto load_v = [&](int kt) __attribute__((always_inline)) {
        const int g = wave / VW;
        const int first = kt * KEYS + 32 * (g >> 2) + 16 * ((g >> 1) & 1) + 4 * (g & 1);  // (uniform)
        const uint32_t off = (uint32_t)my_lane() * 4u;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int key = first + 8 * (e >> 2) + (e & 3);
            const float *row = V + (int64_t)(key < seq_k ? key : seq_k - 1) * d.v_row_stride + (wave % VW) * 64;
            vreg[e] = *reinterpret_cast<const float *>(reinterpret_cast<const char *>(row) + off);
        }
    };
    auto store_k = [&](int kt) __attribute__((always_inline)) {
        float x[8];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            x[e] = kreg[0][e];
            x[4 + e] = kreg[1][e];
        }
#pragma unroll
        for (int e = 0; e < 8; e += 2) k_max = __builtin_fmaxf(__builtin_fmaxf(k_max, __builtin_fabsf(x[e])), __builtin_fabsf(x[e + 1]));
        u32x4 w[kPlanes];
        fth::split8(x, w);
        const int l = my_lane(), kc = l % RL;
        unsigned char *dst = smem + (kt & 1) * STAGE + ((kc * KEYS + ((wave * KROWS + l / RL) ^ (kc << XS))) << 4);
#pragma unroll
        for (int part = 0; part < kPlanes; ++part) *reinterpret_cast<u32x4 *>(dst + part * PART) = w[part];
    };
    auto store_v = [&](int kt) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint32_t u = (__builtin_bit_cast(uint32_t, vreg[e]) << 1) - 1u;  // (zero wraps round)
            v_min = u < v_min ? u : v_min;
        }
#pragma unroll
        for (int e = 0; e < 8; e += 2) v_max = __builtin_fmaxf(__builtin_fmaxf(v_max, __builtin_fabsf(vreg[e])), __builtin_fabsf(vreg[e + 1]));
        u32x4 w[kPlanes];
        fth::split8(vreg, w);
        unsigned char *dst = smem + (kt & 1) * STAGE + VOFF + ((wave / VW * D + (wave % VW) * 64 + my_lane()) << 4);
#pragma unroll
        for (int part = 0; part < kPlanes; ++part) *reinterpret_cast<u32x4 *>(dst + part * PART) = w[part];
    };

    Acc16 o[NDT];
#pragma unroll
    for (int e = 0; e < NDT; ++e)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[e][r] = 0.f;
    float m_run = -__builtin_inff(), l_run = 0.f;

    if (tid < 2) flags[tid] = 0;
    load_k(0);
    store_k(0);
    __syncthreads();

    // Wavefronts 0 - 3 and 4 - 7, one of each on a SIMD, take turns: while one half multiplies (V . P of a stage, then K . Q of the
    // next) the other weighs, so the matrix unit always has a wavefront to feed it and the vector instructions run in its shadow.
    // The second half is half a stage behind and therefore provides its chunks of K and V one stage ahead of the first.
    const int turn = wave >> 2;
    // (past the last stage the last one is read again: a load that may not happen would keep its registers through the loop)
    auto request_k = [&](int kt) __attribute__((always_inline)) { load_k(kt + 1 + turn < num_kt ? kt + 1 + turn : num_kt - 1); };
    auto request_v = [&](int kt) __attribute__((always_inline)) { load_v(kt + turn < num_kt ? kt + turn : num_kt - 1); };
    auto provide = [&](int kt) __attribute__((always_inline)) {
        if (kt + 1 + turn < num_kt) store_k(kt + 1 + turn);
        if (kt + turn < num_kt) store_v(kt + turn);
    };
    if (turn) {
        request_k(-1);
        request_v(-1);
        provide(-1);
        __syncthreads();
    }
    for (int kt = 0; kt < num_kt; ++kt) {
        const int key0 = kt * KEYS + 32 * SUB * kw;
        const bool active = (!d.causal || key0 <= wave_last_q) && key0 < seq_k;
        Acc16 s[SUB];                // scores
        bf16x8 w[2 * SUB][kPlanes];  // parts of the weights
        bf16x8 f[kPlanes];           // operand parts: read again as soon as the last MFMA that takes them is issued
        request_k(kt);
        if constexpr (D == 64) request_v(kt);
        if (active) {
            const unsigned char *s0 = smem + (kt & 1) * STAGE;
            const int l = my_lane(), at = (l >> 5) * KEYS * 16 + (((l & 31) ^ ((l >> 5) << XS)) << 4);
            auto k_read = [&](int i, int part, int to = -1) __attribute__((always_inline)) {
                const int j = i / KSTEPS, t = i % KSTEPS;
                f[to < 0 ? part : to] = *reinterpret_cast<const bf16x8 *>(s0 + (at ^ ((2 * t << XS) << 4)) + 2 * t * KEYS * 16 + (j + SUB * kw) * 512 + part * PART);
            };
#pragma unroll
            for (int j = 0; j < SUB; ++j) {
#pragma unroll
                for (int r = 0; r < 16; ++r) s[j][r] = 0.f;
                k_read(j * KSTEPS, 1);
                k_read(j * KSTEPS, 2);
                k_read(j * KSTEPS, 0);
#pragma unroll
                for (int t = 0; t < KSTEPS; ++t) {  // the lower products of all d ...
                    const int i = j * KSTEPS + t;
                    s[j] = mfma(f[1], q1[t], s[j]);
                    s[j] = mfma(f[1], q0[t], s[j]);
                    __builtin_amdgcn_sched_barrier(0);
                    if (t + 1 < KSTEPS) k_read(i + 1, 1);
                    else k_read(j * KSTEPS, 0, 1);
                    s[j] = mfma(f[2], q0[t], s[j]);
                    __builtin_amdgcn_sched_barrier(0);
                    if (t + 1 < KSTEPS) k_read(i + 1, 2);
                    else k_read(j * KSTEPS + 1, 0, 2);
                    s[j] = mfma(f[0], q2[t], s[j]);
                    s[j] = mfma(f[0], q1[t], s[j]);
                    __builtin_amdgcn_sched_barrier(0);
                    if (t + 1 < KSTEPS) k_read(i + 1, 0);
                    else k_read(j * KSTEPS + 2, 0, 0);
                }
#pragma unroll
                for (int t = 0; t < KSTEPS; ++t) {  // ... then the leading one
                    s[j] = mfma(f[(t + 1) % 3], q0[t], s[j]);
                    __builtin_amdgcn_sched_barrier(0);
                    if (t + 3 < KSTEPS) k_read(j * KSTEPS + t + 3, 0, (t + 1) % 3);
                }
            }
        }
        __syncthreads();
        if constexpr (D == 128) request_v(kt);  // (no registers for it before)
        if (active) {
            constexpr int kMine = 32 * SUB;
            if ((d.causal && key0 + kMine - 1 > q_wave0) || key0 + kMine > seq_k) {
                const int l = my_lane();
                int limit = d.causal ? q_wave0 + (l & 31) : seq_k - 1;  // the last key this query sees
                limit = (limit < seq_k ? limit : seq_k - 1) - key0 - 4 * (l >> 5);
#pragma unroll
                for (int j = 0; j < SUB; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const bool hidden = 32 * j + 8 * (r >> 2) + (r & 3) > limit;
                        s[j][r] = hidden ? -__builtin_inff() : s[j][r];
                    }
            }
            float mt = -__builtin_inff();
#pragma unroll
            for (int j = 0; j < SUB; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) mt = __builtin_fmaxf(mt, s[j][r]);
            // (m is a raw score: the weight of a row's only key is then exactly one)
            if (__any((mt - m_run) * c2 > kLazy)) {
                float mlo, mhi;
                fth::both_halves(mt, mlo, mhi);
                const float m_new = __builtin_fmaxf(m_run, __builtin_fmaxf(mlo, mhi));
                const float alpha = __builtin_amdgcn_exp2f((m_run - m_new) * c2);
#pragma unroll
                for (int e = 0; e < NDT; ++e)
#pragma unroll
                    for (int r = 0; r < 16; ++r) o[e][r] *= alpha;
                l_run *= alpha;
                m_run = m_new;
            }
            float psum = 0.f;
#pragma unroll
            for (int t = 0; t < 2 * SUB; ++t) {
                float x[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    x[e] = __builtin_amdgcn_exp2f((s[t >> 1][8 * (t & 1) + e] - m_run) * c2);
                    psum += x[e];
                }
                u32x4 parts[kPlanes];
                fth::split8(x, parts);
#pragma unroll
                for (int part = 0; part < kPlanes; ++part) w[t][part] = as_bf16(parts[part]);
            }
            l_run += psum;
        }
        provide(kt);
        __syncthreads();
        if (active) {
            const int l = my_lane();
            const unsigned char *s0 = smem + (kt & 1) * STAGE + VOFF + (((l >> 5) * D + (l & 31)) << 4);
            auto v_read = [&](int i, int part) __attribute__((always_inline)) {
                const int e = i / (2 * SUB), t = i % (2 * SUB);
                f[part] = *reinterpret_cast<const bf16x8 *>(s0 + part * PART + (((4 * SUB * kw + 2 * t) * D + 32 * e) << 4));
            };
            v_read(0, 1);
            v_read(0, 2);
            v_read(0, 0);
#pragma unroll
            for (int i = 0; i < NDT * 2 * SUB; ++i) {
                const int e = i / (2 * SUB), t = i % (2 * SUB);
                const bool more = i + 1 < 2 * SUB * NDT;
                o[e] = mfma(f[1], w[t][1], o[e]);
                o[e] = mfma(f[1], w[t][0], o[e]);
                __builtin_amdgcn_sched_barrier(0);
                if (more) v_read(i + 1, 1);
                o[e] = mfma(f[2], w[t][0], o[e]);
                __builtin_amdgcn_sched_barrier(0);
                if (more) v_read(i + 1, 2);
                o[e] = mfma(f[0], w[t][2], o[e]);
                o[e] = mfma(f[0], w[t][1], o[e]);
                o[e] = mfma(f[0], w[t][0], o[e]);
                __builtin_amdgcn_sched_barrier(0);
                if (more) v_read(i + 1, 0);
            }
        }
    }
    __syncthreads();
    if (!turn) __syncthreads();

    // ---- what the parts could not stand for ----
    {
        const bool large = __builtin_amdgcn_ballot_w64(!(k_max < kLarge)) != 0, tiny = __builtin_amdgcn_ballot_w64(v_min < 2 * kTinyBits - 1u) != 0;
        v_max = wave_max(v_max);
        if (lane == 0) {
            if (large) flags[0] = 1;
            if (tiny) flags[1] = 1;
            largest[wave] = v_max;
        }
    }
    if constexpr (KW == 2) {
        // ---- merge the two key halves of each query wavefront (fixed order: half 0, then half 1) ----
        float *mg = reinterpret_cast<float *>(smem) + qw * ((NDT * 16 + 2) * 64) + lane;
        if (kw == 1) {
#pragma unroll
            for (int e = 0; e < NDT; ++e)
#pragma unroll
                for (int r = 0; r < 16; ++r) mg[(e * 16 + r) * 64] = o[e][r];
            mg[(NDT * 16) * 64] = m_run;
            mg[(NDT * 16 + 1) * 64] = l_run;
        }
        __syncthreads();
        if (kw == 1) return;
        const float m1 = mg[(NDT * 16) * 64], l1 = mg[(NDT * 16 + 1) * 64];
        const float m = __builtin_fmaxf(m_run, m1);
        const float a0 = m_run == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f((m_run - m) * c2);
        const float a1 = m1 == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f((m1 - m) * c2);
#pragma unroll
        for (int e = 0; e < NDT; ++e)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[e][r] = o[e][r] * a0 + mg[(e * 16 + r) * 64] * a1;
        l_run = l_run * a0 + l1 * a1;
    } else {
        __syncthreads();
    }
    {
        float llo, lhi;
        fth::both_halves(l_run, llo, lhi);
        l_run = llo + lhi;
    }
    float big = 0.f, small = FLT_MAX;
#pragma unroll
    for (int e = 0; e < NDT; ++e)
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
            o[e][r] = o[e][r] / l_run;
            o[e][r + 1] = o[e][r + 1] / l_run;
            const float a = __builtin_fabsf(o[e][r]), b = __builtin_fabsf(o[e][r + 1]);
            big = nan_max(nan_max(big, a), b);
            small = __builtin_fminf(__builtin_fminf(small, a), b);
        }
    bool doubt = !(big <= FLT_MAX) || q_large || flags[0] != 0 || (flags[1] != 0 && small < kTinyOut);
    float share = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) share = __builtin_fmaxf(share, largest[w]);
    share = __builtin_fminf(share, FLT_MAX) * kTinyShare;
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(small < share) != 0, 0)) {  // (zeros do not count)
#pragma unroll
        for (int e = 0; e < NDT; ++e)
#pragma unroll
            for (int r = 0; r < 16; ++r) doubt |= o[e][r] != 0.f && __builtin_fabsf(o[e][r]) < share;
    }
    doubt &= q_live;
    if (__builtin_amdgcn_ballot_w64(doubt)) {
        const int k_last = d.causal && wave_last_q + 1 < seq_k ? wave_last_q + 1 : seq_k;
        Acc16 f[NDT];
        fth::sdpa_rows_f32<D>(d, Q, K, V, c2, q_wave0, (k_last + 31) / 32, f, l_run);
        if (q_live) {
            float *orow = O + (int64_t)qi * d.o_row_stride;
#pragma unroll
            for (int r = 0; r < 16; ++r)
#pragma unroll
                for (int e = 0; e < NDT; ++e) orow[NDT * (8 * (r >> 2) + 4 * half + (r & 3)) + e] = f[e][r] / l_run;
        }
        return;
    }
    // ---- lane owns query qi, d = 32 e + 8 (r / 4) + 4 half + r % 4 ----
    if (q_live) {
        float *orow = O + (int64_t)qi * d.o_row_stride + 4 * half;
#pragma unroll
        for (int e = 0; e < NDT; ++e)
#pragma unroll
            for (int g = 0; g < 4; ++g) *reinterpret_cast<f32x4 *>(orow + 32 * e + 8 * g) = f32x4{o[e][4 * g], o[e][4 * g + 1], o[e][4 * g + 2], o[e][4 * g + 3]};
    }
}

template <int D, int QW, int KW> int32_t launch(SplitSdpaArgs &a, hipStream_t st) {
    constexpr int smem = 2 * 2 * fth::kPlanes * 4096 * 2;
    auto kern = sdpa_split_kernel<D, QW, KW>;
    static const hipError_t ready = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    FTH_HIP(ready);
    a.q_blocks = (int)fth::ceil_div(a.d.seq_q, 32 * QW);
    const int64_t grid = a.d.num_bh * a.q_blocks;
    FTH_ARG(grid <= 2147483647LL, "sdpa: grid too large");
    kern<<<dim3((unsigned)grid), dim3(64 * QW * KW), smem, st>>>(a);
    FTH_CHECK_LAUNCH("sdpa_split");
    return FTH_OK;
}

int forced_config() {
    static const int v = [] {
        const char *e = std::getenv("FT_HIP_SDPA_SPLIT");  // tuning knob: 0 keeps attention on fp32 MFMAs, 1 / 2 force 256 queries a workgroup / 128 and two key halves
        const char *cfg = std::getenv("FT_HIP_SDPA_CFG");  // (a forced configuration of the fp32 kernel means that kernel)
        return cfg && std::atoi(cfg) >= 0 ? 0 : e ? std::atoi(e) : -1;
    }();
    return v;
}

// Head size 64 has two forms. Time of a launch in stages of 64 keys by 256 queries: whole rounds of workgroups, or for causal
// problems, which are issued longest first, the average load and a third of the longest block, but no less than that one. A stage
// of the 128-query form takes 0.64 of the other's time (0.58 with every compute unit busy, 0.65 with few): measured over 144
// problems of 8 to 128 heads and 128 to 2048 tokens this picks the faster form, or one at most 6% slower.
double stages(const fth_sdpa_desc &d, int block, double stage) {
    const int cus = fth::compute_units() > 0 ? fth::compute_units() : 256;
    const int64_t blocks = fth::ceil_div(d.seq_q, (int64_t)block), whole = fth::ceil_div(d.seq_k, 64);
    if (!d.causal) return (double)fth::ceil_div(d.num_bh * blocks, (int64_t)cus) * whole * stage;
    // block i (of `blocks`) sees min((i + 1) block, seq_k) keys: a ramp up to the first block that sees all of them, then level
    const int64_t per = block / 64, ramp = whole / per < blocks ? whole / per : blocks;
    const double total = (double)per * ramp * (ramp + 1) / 2 + (double)(blocks - ramp) * whole;
    const double longest = (double)(whole < per * blocks ? whole : per * blocks);
    const double load = total * d.num_bh / cus + 0.33 * longest;
    return (load > longest ? load : longest) * stage;
}

}  // namespace

namespace fth {

bool sdpa_split_pays(const fth_sdpa_desc &d, float scale) {
    if (forced_config() == 0 || d.d_k != d.d_v || (d.d_k != 64 && d.d_k != 128) || d.k_row_stride < 0 || d.v_row_stride < 0 ||
        !(scale > 0.f && scale <= 0x1p20f) || d.seq_k < 1)
        return false;
    // Head size 128: with few keys, or only half of a block's queries on a full chip, the fp32 kernel is as fast or faster (us there
    // / here: 8 heads x 9 queries x 9 keys 10.3 / 11.4, 200 x 128 22.6 / 24.1, 256 heads x 100 x 2048 262 / 269; on this side 8 heads
    // of 200 x 200 34.4 / 31.2, 64 heads of 100 x 2048 and above).
    const int64_t keys = d.causal && d.seq_q < d.seq_k ? d.seq_q : d.seq_k;
    if (d.d_k == 128 && (keys < 160 || (d.seq_q <= 128 && d.num_bh > 128))) return false;
    // Head size 64: one stage of keys leaves nothing to hide a block's start and end behind, and the fp32 kernel is the faster one where blocks that
    // are half empty at the least take a second round here (260 heads x 64 x 64 13.4 / 16.6, 512 x 48 x 64 14.3 / 17.2, 1024 x 64 x 64 causal
    // 20.2 / 35.4, 260 x 100 x 64 14.9 / 18.1; in one, 192 x 48 x 48 9.9 / 9.2). Longer ones stay for their smaller error (1.2e-7, there 2.4e-7),
    // on either side in time: 96 x 300 x 40 15.8 / 12.6, 128 x 600 x 64 24.9 / 28.7, 32 x 300 x 64 9.0 / 10.3. With more keys: 260 x 64 x 100 22.3 /
    // 21.6, 768 x 127 x 127 causal 39.1 / 38.6.
    const int64_t cus = compute_units() > 0 ? compute_units() : 256;
    if (d.d_k == 64 && keys <= 64 && d.seq_q <= 128 && d.num_bh > cus) return false;
    // Head size 128, not causal: a second round of 256-query blocks where all blocks of the fp32 kernel, 128 queries and two on a
    // compute unit, run at once (96 heads x 640 tokens: 172 us, 165 there).
    if (d.d_k == 128 && !d.causal && d.num_bh * ceil_div(d.seq_q, (int64_t)256) > cus && d.num_bh * ceil_div(d.seq_q, (int64_t)128) <= 2 * cus) return false;
    return true;
}

int32_t sdpa_split_f32(const fth_sdpa_desc &d, float scale, const float *q, const float *k, const float *v, float *out, hipStream_t st) {
    SplitSdpaArgs a{q, k, v, out, d, scale, 0, d.kv_group > 1 ? d.kv_group : 1};
    if (d.d_k == 128) return launch<128, 8, 1>(a, st);
    const int forced = forced_config();
    const bool halves = forced > 0 ? forced == 2 : stages(d, 128, 0.64) < stages(d, 256, 1.0);
    return halves ? launch<64, 4, 2>(a, st) : launch<64, 8, 1>(a, st);
}

}  // namespace fth
