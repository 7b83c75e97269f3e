// Attention of a few new tokens per sequence against a long K/V cache (seq_q <= 8, no causal flag), fp32.
//
// Bound by reading K and V once: 4 D flops per K/V element and query row are nothing beside 8 bytes of cache per element
// pair. So the split of the work is by keys, and all query rows that share a K/V head (group x seq_q of them) ride on one
// pass over it:
//   * a wavefront owns up to 16 (QT = 1) or 32 (QT = 2) query rows of one K/V head and one contiguous share of the keys, and
//     walks it in tiles of 32 keys with an online softmax; nothing goes through LDS and no wavefront waits for another;
//   * S^T[key, row] = K . Q^T on v_mfma_f32_16x16x4_f32: a lane's A operand is one K row read as float4s (two consecutive
//     ones, so that the four lanes of a row cover a whole 128-byte line), its B operand one query row held in registers. The
//     lane that gets a score then holds it as the B operand of O^T[d, row] += V^T . P^T, so P never moves; V rows are read
//     whole, D / 16 consecutive floats per lane;
//   * the K loads of the next tile are issued as soon as the scores have consumed this one's, the V loads before the scores,
//     so both are in flight under the softmax;
//   * the shares of a row are merged by a second small kernel in key order (partial maximum, sum and unnormalised output).
// The number of shares depends on (num_bh, seq_k), the head size and whether there is a mask -- not on how many query heads
// share a K/V head -- so a grouped call and the same call on repeated K/V heads give the same bits.
// Rows past group x seq_q are padding (the matrix pipe runs at 0.3 of its rate even for one row of 16, under the loads).
//
// Measured at 16 sequences, 32 query heads on 8 K/V heads, 3967 keys, D 128, per-row mask (529 MB): 1108 us on the 128-query
// kernel, 113 us here (4.7 TB/s); 14 sequences, 278 keys, D 64: 70 -> 16 us.
//
// Semantics of sdpa_forward_f32 / sdpa_forward_masked_f64 (crates/ft-kernel-cpu/src/lib.rs:5200-5284, 4661-4741): scale after
// the product, additive mask, softmax over all keys; a row with every key hidden is NaN.

#include <optional>
#include <type_traits>

#include "common.hpp"
#include "sdpa_decode.hpp"
#include "stream_scratch.hpp"

namespace {

using Acc4 = float __attribute__((ext_vector_type(4)));
using F4 = float __attribute__((ext_vector_type(4)));
using F4u = float __attribute__((ext_vector_type(4), aligned(4)));  // mask rows start anywhere

constexpr int kTile = 32;  // keys per step: two 16-key MFMA tiles

struct DecodeArgs {
    const float *q, *k, *v, *mask;
    float *out;
    float *part_o;   // [unit][split][16 QT][D] unnormalised outputs (more than one share)
    float *part_ml;  // [unit][split][16 QT][2] running maximum and sum
    fth_sdpa_desc d;
    float scale;
    int64_t mask_bh_stride;
    int group, kv_heads, row_tiles, nsplit, tiles_per_split;
};

// max / sum over the four 16-lane rows of a wavefront, the result in every lane (two register swaps, no LDS)
template <typename F> __device__ __forceinline__ float rows_reduce(float x, F op) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = op(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return op(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

template <int NE> struct VRow {  // NE consecutive floats of a V row
    F4 v[NE / 4];
    __device__ __forceinline__ void load(const float *p) {
#pragma unroll
        for (int i = 0; i < NE / 4; ++i) v[i] = reinterpret_cast<const F4 *>(p)[i];
    }
    __device__ __forceinline__ float get(int e) const { return v[e / 4][e % 4]; }
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int i = 0; i < NE / 4; ++i) v[i] = F4{0.f, 0.f, 0.f, 0.f};
    }
};
template <> struct VRow<2> {
    float2 v;
    __device__ __forceinline__ void load(const float *p) { v = *reinterpret_cast<const float2 *>(p); }
    __device__ __forceinline__ float get(int e) const { return e == 0 ? v.x : v.y; }
    __device__ __forceinline__ void clear() { v = make_float2(0.f, 0.f); }
};

template <int D, int QT, bool MASK>
__global__ __launch_bounds__(64, QT == 1 ? 2 : 1) void sdpa_decode_kernel(const DecodeArgs p) {
    constexpr int NT = D / 16;  // float4s of a K row per lane
    constexpr int NE = D / 16;  // consecutive output columns per lane and MFMA row
    constexpr int ROWS = 16 * QT;
    const int lane = threadIdx.x, lr = lane & 15, g = lane >> 4;
    const int split = (int)(blockIdx.x % (unsigned)p.nsplit);
    const int64_t unit = blockIdx.x / (unsigned)p.nsplit;
    const int rt = (int)(unit % p.row_tiles);
    const int64_t bk = unit / p.row_tiles;  // batch * kv_heads + K/V head
    const int64_t batch = bk / p.kv_heads;
    const int hk = (int)(bk % p.kv_heads);
    const int seq_q = (int)p.d.seq_q, seq_k = (int)p.d.seq_k, rows = p.group * seq_q;
    const float *K = p.k + batch * p.d.k_batch_stride + hk * p.d.k_head_stride;
    const float *V = p.v + batch * p.d.v_batch_stride + hk * p.d.v_head_stride;

    F4 q[QT][NT];
    const float *mrow[QT];
#pragma unroll
    for (int t = 0; t < QT; ++t) {
        int rr = rt * ROWS + t * 16 + lr;
        rr = rr < rows ? rr : rows - 1;  // padding rows repeat the last one; they are never stored
        const int h = hk * p.group + rr / seq_q, qi = rr % seq_q;
        const float *qr = p.q + batch * p.d.q_batch_stride + h * p.d.q_head_stride + qi * p.d.q_row_stride + 8 * g;
#pragma unroll
        for (int i = 0; i < NT; ++i) q[t][i] = *reinterpret_cast<const F4 *>(qr + 32 * (i >> 1) + 4 * (i & 1));
        mrow[t] = MASK ? p.mask + (batch * p.d.heads + h) * p.mask_bh_stride + (int64_t)qi * seq_k : nullptr;
    }

    const int key_lo = split * p.tiles_per_split * kTile;
    int key_hi = key_lo + p.tiles_per_split * kTile;
    key_hi = key_hi < seq_k ? key_hi : seq_k;
    const unsigned ks = (unsigned)p.d.k_row_stride, vs = (unsigned)p.d.v_row_stride;  // seq_k * stride fits 30 bits (launcher check)

    F4 kf[2][NT];
    auto load_k = [&](int key0) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            int key = key0 + 16 * s + lr;
            key = key < seq_k ? key : seq_k - 1;  // keys past the end are weighted zero
            const float *kr = K + ((unsigned)key * ks + 8u * (unsigned)g);
#pragma unroll
            for (int i = 0; i < NT; ++i) kf[s][i] = *reinterpret_cast<const F4 *>(kr + 32 * (i >> 1) + 4 * (i & 1));
        }
    };

    Acc4 o[QT][NE];
    float m_run[QT], l_run[QT];
#pragma unroll
    for (int t = 0; t < QT; ++t) {
        m_run[t] = -__builtin_inff();
        l_run[t] = 0.f;  // this lane's share of the row sum; the four lanes of a row are added at the end
#pragma unroll
        for (int e = 0; e < NE; ++e) o[t][e] = Acc4{0.f, 0.f, 0.f, 0.f};
    }

    if (key_lo < key_hi) load_k(key_lo);
    for (int key0 = key_lo; key0 < key_hi; key0 += kTile) {
        VRow<NE> vf[2][4];
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                int key = key0 + 16 * s + 4 * g + r;
                key = key < seq_k ? key : seq_k - 1;
                vf[s][r].load(V + ((unsigned)key * vs + (unsigned)(lr * NE)));
            }
        F4u mk[QT][2];
        if constexpr (MASK) {
#pragma unroll
            for (int t = 0; t < QT; ++t)
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const int key = key0 + 16 * s + 4 * g;
                    if (key + 3 < seq_k) mk[t][s] = *reinterpret_cast<const F4u *>(mrow[t] + key);
                    else
#pragma unroll
                        for (int r = 0; r < 4; ++r) mk[t][s][r] = key + r < seq_k ? mrow[t][key + r] : 0.f;
                }
        }
        Acc4 sc[QT][2];
#pragma unroll
        for (int t = 0; t < QT; ++t)
#pragma unroll
            for (int s = 0; s < 2; ++s) sc[t][s] = Acc4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int t = 0; t < QT; ++t)
#pragma unroll
                    for (int s = 0; s < 2; ++s) sc[t][s] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[s][i][j], q[t][i][j], sc[t][s], 0, 0, 0);
        if (key0 + kTile < key_hi) load_k(key0 + kTile);
        // online softmax: a lane holds keys 16 s + 4 g + r of row lr
#pragma unroll
        for (int t = 0; t < QT; ++t) {
            float mx = -__builtin_inff();
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float x = sc[t][s][r] * p.scale;
                    if constexpr (MASK) x = x + mk[t][s][r];
                    if (key0 + 16 * s + 4 * g + r >= key_hi) x = -__builtin_inff();
                    sc[t][s][r] = x;
                    mx = fmaxf(mx, x);
                }
            mx = rows_reduce(mx, [](float a, float b) { return fmaxf(a, b); });
            const float m_new = fmaxf(m_run[t], mx);
            const float m_ref = m_new == -__builtin_inff() ? 0.f : m_new;  // nothing visible so far: every weight is exp(-inf) = 0
            const float alpha = __builtin_amdgcn_exp2f((m_run[t] - m_ref) * 1.44269502162933349609375f);
            m_run[t] = m_new;
            float sum = 0.f;
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float e = __builtin_amdgcn_exp2f((sc[t][s][r] - m_ref) * 1.44269502162933349609375f);
                    sc[t][s][r] = e;
                    sum += e;
                }
            l_run[t] = l_run[t] * alpha + sum;
#pragma unroll
            for (int e = 0; e < NE; ++e)
#pragma unroll
                for (int r = 0; r < 4; ++r) o[t][e][r] *= alpha;
        }
        if (key0 + kTile > seq_k) {  // weight 0 times an infinite value would be NaN
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (key0 + 16 * s + 4 * g + r >= seq_k) vf[s][r].clear();
        }
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int e = 0; e < NE; ++e)
#pragma unroll
                    for (int t = 0; t < QT; ++t)
                        o[t][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[s][r].get(e), sc[t][s][r], o[t][e], 0, 0, 0);
    }

#pragma unroll
    for (int t = 0; t < QT; ++t) {
        const float l = rows_reduce(l_run[t], [](float a, float b) { return a + b; });
        const int rr = rt * ROWS + t * 16 + lr;
        if (rr >= rows) continue;
        float *dst;
        if (p.nsplit == 1) {
            const int h = hk * p.group + rr / seq_q, qi = rr % seq_q;
            dst = p.out + batch * p.d.o_batch_stride + h * p.d.o_head_stride + qi * p.d.o_row_stride;
        } else {
            const int64_t slot = (unit * p.nsplit + split) * ROWS + t * 16 + lr;
            dst = p.part_o + slot * D;
            if (g == 0) {
                p.part_ml[2 * slot] = m_run[t];
                p.part_ml[2 * slot + 1] = l;
            }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r)  // MFMA row 4 g + r of column tile e is output column (4 g + r) NE + e
#pragma unroll
            for (int e = 0; e < NE; ++e) dst[(4 * g + r) * NE + e] = p.nsplit == 1 ? o[t][e][r] / l : o[t][e][r];
    }
}

// out = sum_s w_s O_s / sum_s w_s l_s with w_s = exp(m_s - max m), shares in key order. One thread per four output columns.
template <int D, int QT> __global__ __launch_bounds__(256) void sdpa_decode_merge_kernel(const DecodeArgs p) {
    constexpr int ROWS = 16 * QT, V4 = D / 4;
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int c = (int)(idx % V4);
    const int64_t row = idx / V4;  // bh * seq_q + qi
    if (row >= p.d.num_bh * p.d.seq_q) return;
    const int seq_q = (int)p.d.seq_q;
    const int64_t bh = row / seq_q;
    const int qi = (int)(row % seq_q);
    const int64_t batch = bh / p.d.heads;
    const int h = (int)(bh % p.d.heads), hk = h / p.group;
    const int rr = (h % p.group) * seq_q + qi;
    const int64_t unit = (batch * p.kv_heads + hk) * p.row_tiles + rr / ROWS;
    const int64_t slot0 = unit * p.nsplit * ROWS + rr % ROWS;
    float m = -__builtin_inff();
    for (int s = 0; s < p.nsplit; ++s) m = fmaxf(m, p.part_ml[2 * (slot0 + (int64_t)s * ROWS)]);
    const float m_ref = m == -__builtin_inff() ? 0.f : m;
    F4 acc = {0.f, 0.f, 0.f, 0.f};
    float l = 0.f;
#pragma unroll 4
    for (int s = 0; s < p.nsplit; ++s) {
        const int64_t slot = slot0 + (int64_t)s * ROWS;
        const float w = __builtin_amdgcn_exp2f((p.part_ml[2 * slot] - m_ref) * 1.44269502162933349609375f);
        const F4 o = *reinterpret_cast<const F4 *>(p.part_o + slot * D + 4 * c);
        l += p.part_ml[2 * slot + 1] * w;
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] += o[i] * w;
    }
    F4 y;
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] = acc[i] / l;
    *reinterpret_cast<F4 *>(p.out + batch * p.d.o_batch_stride + h * p.d.o_head_stride + qi * p.d.o_row_stride + 4 * c) = y;
}

// *done stays false, with nothing launched, when the grid or the scratch memory cannot be had.
template <int D, int QT> int32_t launch(DecodeArgs &a, hipStream_t st, bool *done) {
    constexpr int ROWS = 16 * QT;
    a.row_tiles = (int)fth::ceil_div((int64_t)a.group * a.d.seq_q, ROWS);
    const int64_t units = a.d.num_bh / a.group * a.row_tiles;
    const int64_t grid = units * a.nsplit;
    if (grid > 2147483647LL) return FTH_OK;
    std::optional<fth::StreamScratch> lease;  // until the merge is queued
    if (a.nsplit > 1) {
        const int64_t slots = grid * ROWS;
        void *ws = lease.emplace().get(st, fth::ScratchUse::DecodeShares, (size_t)(slots * (D + 2)) * sizeof(float));
        if (!ws) return FTH_OK;
        a.part_o = static_cast<float *>(ws);
        a.part_ml = a.part_o + slots * D;
    }
    *done = true;
    if (a.mask) sdpa_decode_kernel<D, QT, true><<<dim3((unsigned)grid), dim3(64), 0, st>>>(a);
    else sdpa_decode_kernel<D, QT, false><<<dim3((unsigned)grid), dim3(64), 0, st>>>(a);
    FTH_CHECK_LAUNCH("sdpa_decode");
    if (a.nsplit > 1) {
        const int64_t n = a.d.num_bh * a.d.seq_q * (D / 4);
        sdpa_decode_merge_kernel<D, QT><<<dim3((unsigned)fth::ceil_div(n, 256)), dim3(256), 0, st>>>(a);
        FTH_CHECK_LAUNCH("sdpa_decode_merge");
    }
    return FTH_OK;
}

template <int D> int32_t launch_rows(DecodeArgs &a, hipStream_t st, bool *done) {
    // Row tiles of 16 where the rows fit one, and up to 2048 keys (more tiles, which the chip has room for: 32 query heads on 8
    // K/V heads, 8 queries, 128 keys of 64: 11.9 -> 9.4 us); else of 32, which read K and V half as often (4096 keys: 34 against
    // 36 us). A row is computed alike in both.
    return (int64_t)a.group * a.d.seq_q <= 16 || a.d.seq_k <= 2048 ? launch<D, 1>(a, st, done) : launch<D, 2>(a, st, done);
}

}  // namespace

namespace fth {

// seq_q <= 8: the tiled kernels of csrc/sdpa.hip pad to 128 queries and read K and V once per query head: 2 times slower at 16
// keys, 4 to 10 times at 4096. Its key-split kernel for small problems (short_alternative: it would take the call otherwise)
// needs one launch where this one needs a second for the merge, and is the faster one past the 64 keys of a single share while K
// is short. us, that kernel / this one, 12 heads of 64, one query: 64 keys 7.6 / 5.8, 128 keys 7.9 / 9.2, 256 keys 10.9 / 9.6,
// 4096 keys 97 / 32; of 32: 256 keys 7.5 / 8.1, 512 keys 11.0 / 9.3. With more than 128 query heads and 5 to 8 queries the line
// is at twice that (256 heads, 384 keys of 64: 14.9 / 18.6). Neither the number of K/V heads nor that of shares decides, so a
// grouped call and the same call on repeated K/V heads take the same path; the price is up to a tenth on 192 to 256 ungrouped
// heads of up to 1024 keys (512 keys of 64: 18.9 / 19.9), where grouped ones gain a third to a half.
bool sdpa_decode_applies(const fth_sdpa_desc &d, bool short_alternative) {
    const int64_t line = d.num_bh > 128 && d.seq_q > 4 ? 32768 : 16384;
    if (short_alternative && d.seq_k > 64 && d.seq_k * d.d_k < line) return false;
    // a head's K and V are addressed through unsigned 32-bit offsets, key numbers are ints with room for the last share
    auto span_ok = [&](int64_t row_stride) { return row_stride >= 0 && d.seq_k * row_stride < ((int64_t)1 << 30); };
    return d.causal == 0 && d.seq_q <= 8 && d.seq_k > 0 && d.seq_k <= ((int64_t)1 << 28) && d.d_k == d.d_v &&
           (d.d_k == 128 || d.d_k == 64 || d.d_k == 32) && span_ok(d.k_row_stride) && span_ok(d.v_row_stride);
}

bool sdpa_decode_f32(const fth_sdpa_desc &d, float scale, const float *q, const float *k, const float *v, const float *mask,
                     int64_t mask_bh_stride, float *out, bool short_alternative, hipStream_t st, int32_t *rc) {
    DecodeArgs a;
    a.q = q; a.k = k; a.v = v; a.mask = mask; a.out = out;
    a.part_o = a.part_ml = nullptr;
    a.d = d;
    a.scale = scale;
    a.mask_bh_stride = mask_bh_stride;
    a.group = d.kv_group > 1 ? (int)d.kv_group : 1;
    a.kv_heads = (int)(d.heads / a.group);
    a.row_tiles = 1;
    // Shares of the keys: about 8192 (query head, share) pairs, which is 8 wavefronts per compute unit even where four query
    // heads ride on one K/V head; at least two 32-key tiles per share. Half of that without a mask at head sizes 32 and 64, where
    // the merge weighs more: 256 heads on 256 K/V heads, 2048 keys of 64 62 -> 56 us, on 32 K/V heads 23 -> 18 us (with a mask at
    // head size 128 and 4 queries, 256 heads on 32, 4096 keys it would cost 52 -> 65 us).
    const int64_t tiles = fth::ceil_div(d.seq_k, kTile);
    int64_t want = (short_alternative ? 4096 : 8192) / (d.num_bh > 0 ? d.num_bh : 1);
    const int64_t most = tiles / 2 > 0 ? tiles / 2 : 1;
    want = want < 1 ? 1 : want > most ? most : want;
    a.tiles_per_split = (int)fth::ceil_div(tiles, want);
    a.nsplit = (int)fth::ceil_div(tiles, a.tiles_per_split);
    bool done = false;
    *rc = d.d_k == 128 ? launch_rows<128>(a, st, &done) : d.d_k == 64 ? launch_rows<64>(a, st, &done) : launch_rows<32>(a, st, &done);
    return done;
}

}  // namespace fth
