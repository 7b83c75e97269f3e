// fp32 matrix products on the bf16 matrix units.
//
// Each operand is split into three bf16 parts that sum to it exactly (split_bf16.hpp); six products of parts are formed and summed
// in fp32. Six bf16 MFMAs of 32 k cost 96 cycles where the fp32 MFMAs cost 256. x0 y0 has an accumulator of its own: the other
// five are 2^-8 of it and less, and each of them added to the full sum would round that sum again (several times an MFMA, which
// adds in groups), so they are kept apart until the end of the tile. Relative 2-norm error against 64-bit sums, this kernel / the fp32 MFMA kernel:
//   normal operands, K 768, 3072, 4096, 50257: 1.6e-7 / 4.95e-7, 3.4e-7 / 9.9e-7, 4.0e-7 / 1.15e-6, 3.5e-7 / 1.7e-6
//   of one sign (uniform), the same K:         1.5e-7 / 4.2e-7,  3.0e-7 / 8.3e-7, 3.0e-7 / 8.4e-7,  1.0e-7 / 6.1e-7
//   ReLU of normal, the same K:                1.2e-7 / 3.5e-7,  2.7e-7 / 7.0e-7, 3.2e-7 / 8.1e-7,  2.9e-7 / 1.2e-6
// (With one accumulator for all six: 4.2e-7 / 8.6e-7 / 1.00e-6 / 1.1e-6 on normal operands, and worse than the fp32 kernel by a
// sixth on ReLU ones.) A sum of a single non-zero product is the one place where the left-out terms show: 2.6e-8 / 2.5e-8, the
// largest error 1.7 / 1.0 units of 2^-24.
//
// Two passes. split_kernel writes an operand's three planes once, in the order in which the product
// reads them; the product then moves planes to LDS with direct loads and has no vector arithmetic in its loop. Splitting
// inside the product was tried and costs more: vector instructions and MFMAs share issue cycles, every element would be
// split again by each tile that reads it, and the loop stayed at 190-230 TFLOP/s (of fp32 products) where this one reaches
// 240-264.
//
// What the split cannot stand for is found in the results. Non-zero operands under 2^-110, whose third part would lie below the
// bf16 subnormals, operands of 2^53 and more, whose sums of up to 2^20 products could overflow where fp32 arithmetic does not,
// infinities and NaN are written as NaN planes and leave NaN sums; every other operand is exactly the sum of its parts. In
// a sum under 2^-100 products of the lower parts may have been rounded at the end of the fp32 range (the matrix unit keeps
// subnormals, measured). A wavefront that holds a NaN or a non-zero sum under 2^-100 computes its part of the tile again from
// the fp32 operands on fp32 MFMAs.
//
// replaces gemm::sgemm / sgemm_bt / sgemm_tb (crates/ft-kernel-cpu/src/lib.rs:1310-1338, 1430-1524) for large products.

#include <cfloat>
#include <cstdlib>

#include "common.hpp"
#include "devmath.hpp"
#include "gemm_split.hpp"
#include "split_bf16.hpp"
#include "stream_scratch.hpp"

namespace {

constexpr int kWave = 64;
constexpr int kXcds = 8;
constexpr int kGroupM = 8;
constexpr int kBK = 32;       // k of a K-tile: one 16 x 16 x 32 MFMA
constexpr int kBlock = 1024;  // bytes of one plane of 16 rows x 32 k
constexpr float kTiny = 0x1p-100f;
constexpr uint32_t kTooLarge = 0x5a000000u, kTooSmall = 0x08800000u;  // bits of 2^53 and of 2^-110

using fth::bf16x8;
using fth::f32x4;
using fth::kPlanes;
using fth::u32x4;
typedef f32x4 f32x4_any __attribute__((aligned(4)));  // 128-bit access at any float

// NaN in the place of a float that the parts cannot stand for.
__device__ __forceinline__ float representable(float x) {
    const uint32_t u = __builtin_bit_cast(uint32_t, x) & 0x7fffffffu;
    return u >= kTooLarge || u - 1u < kTooSmall - 1u ? __builtin_nanf("") : x;  // (zero wraps round)
}

// Planes of an operand: [K-tile][plane][16-row block][16 rows][4 chunks of 8 k], a 16-byte chunk at slot chunk ^ fth::swz(row) of
// its row. The LDS holds the same image, and a wavefront's 128-bit operand read (16 rows at the same chunk, in the lane
// groups the LDS serves together) touches every bank once: 0 conflict cycles by counter; chunk ^ (row / 4) has 2 a read.

__device__ __forceinline__ void store_chunk(const float (&v)[8], unsigned char *planes, int64_t kt, int blocks, int64_t row, int chunk) {
    float r[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) r[e] = representable(v[e]);
    u32x4 w[kPlanes];
    fth::split8(r, w);
#pragma unroll
    for (int s = 0; s < kPlanes; ++s)
        *reinterpret_cast<u32x4 *>(planes + (kt * kPlanes + s) * blocks * kBlock + row * 64 + ((chunk ^ fth::swz((int)(row & 15))) << 4)) = w[s];
}

// One operand to split: [rows][k] (by_k) with row pitch ld, or [k][rows] with row pitch ld.
struct SplitArgs {
    const float *x;
    unsigned char *planes;
    int64_t rows, k, ld;
    int blocks, ktiles;  // 16-row blocks, K-tiles
    bool by_k;
    int64_t groups;      // workgroups
};

// Both operands of a product in one launch. Stored [rows][k]: a wavefront takes one 16-row block and one K-tile, whole 128-byte
// lines in, three whole 1 KB blocks out. Stored [k][rows]: a workgroup takes 64 rows and one K-tile, a wavefront one 8-k chunk
// of it, 256-byte runs in. Rows and k beyond the operand are zero. Bound by memory: 4 bytes in, 6 out per element; 103 M
// elements (2048 x 50257) in 200 us, 5.1 TB/s.
__global__ __launch_bounds__(256) void split_kernel(const SplitArgs first, const SplitArgs second) {
    const bool is_first = blockIdx.x < first.groups;
    const SplitArgs &o = is_first ? first : second;
    const int64_t id = is_first ? blockIdx.x : blockIdx.x - first.groups;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float v[8];
    if (o.by_k) {
        const int64_t quads = (o.ktiles + 3) / 4, blk = id / quads, kt = (id - blk * quads) * 4 + wave;
        if (kt >= o.ktiles) return;
        const int64_t row = blk * 16 + (lane >> 2);
        const int chunk = lane & 3;
        const int64_t k0 = kt * kBK + chunk * 8;
        if (row < o.rows && k0 + 8 <= o.k) {
            const float *src = o.x + row * o.ld + k0;
            const f32x4 lo = *reinterpret_cast<const f32x4_any *>(src), hi = *reinterpret_cast<const f32x4_any *>(src + 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = lo[e];
                v[4 + e] = hi[e];
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = row < o.rows && k0 + e < o.k ? o.x[row * o.ld + k0 + e] : 0.f;
        }
        store_chunk(v, o.planes, kt, o.blocks, row, chunk);
    } else {
        const int64_t across = (o.blocks + 3) / 4, kt = id / across, row = (id - kt * across) * 64 + lane, k0 = kt * kBK + wave * 8;
        if (row >= (int64_t)o.blocks * 16) return;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = row < o.rows && k0 + e < o.k ? o.x[(k0 + e) * o.ld + row] : 0.f;
        store_chunk(v, o.planes, kt, o.blocks, row, wave);
    }
}

struct PlaneArgs {
    fth::SplitGemm g;
    const unsigned char *a, *b;
    int a_blocks, b_blocks;  // 16-row blocks of the planes
    int ktiles;              // of the whole product
    int splits, kt_per;      // the K-tiles are cut into `splits` runs of kt_per (the last one shorter)
    int tiles_m, tiles_n;
    int tiles;
    float *partial;          // splits > 1: [splits][m][n] sums without epilogue
    int order;               // tile order inside a group of tile rows, as in the fp32 kernel: 1 walks along the rows of C
    int64_t rowmax_groups;
};

__device__ __forceinline__ void tile_of_id(int id, int tiles_m, int tiles_n, int order, int &tm, int &tn) {
    const int group = kGroupM * tiles_n;
    const int g = id / group;
    const int first_m = g * kGroupM;
    const int gm = (tiles_m - first_m) < kGroupM ? (tiles_m - first_m) : kGroupM;
    const int in_g = id - g * group;
    tm = first_m + (order ? in_g / tiles_n : in_g % gm);
    tn = order ? in_g % tiles_n : in_g / gm;
}

// Hardware workgroup id -> virtual id such that each XCD owns one contiguous run of virtual ids.
__device__ __forceinline__ int xcd_contiguous_id(int pid, int grid) {
    const int per = grid / kXcds, rem = grid % kXcds, xcd = pid % kXcds, q = pid / kXcds;
    return q + xcd * per + (xcd < rem ? xcd : rem);
}

__device__ __forceinline__ const unsigned char *uniform_ptr(const unsigned char *ptr) {
    const uint64_t v = reinterpret_cast<uint64_t>(ptr);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return reinterpret_cast<const unsigned char *>(((uint64_t)hi << 32) | lo);
}

// 1 KB from a uniform base plus per-lane offsets to LDS. In assembly so that the compiler does not wait for it at the next LDS
// read; the kernel waits for vmcnt(0) itself before each barrier. Writes no register.
__device__ __forceinline__ void load_to_lds_16(const unsigned char *base, unsigned lane_bytes, unsigned lds_chunk) {
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(lane_bytes), "s"(base), "s"(lds_chunk) : "memory", "m0");
}

__device__ __forceinline__ float nan_max(float a, float b) { return __builtin_elementwise_maximum(a, b); }

// Four k of one operand row for the fp32 MFMAs: the first `left` of them from p on, ks apart, the others zero.
__device__ __forceinline__ f32x4 four_k(const float *p, int64_t ks, int left) {
    if (ks == 1 && left >= 4) return *reinterpret_cast<const f32x4_any *>(p);
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (e < left) v[e] = p[e * ks];
    return v;
}

// The product. WM x WN wavefronts share a BM x BN tile; a wavefront's operands of one K-tile are 3 (TM + TN) 128-bit LDS reads
// for 6 TM TN MFMAs. Two LDS buffers of a K-tile's planes, one barrier a K-tile: behind it the loads of the K-tile after
// next are issued into the buffer that was just read out, and the operands of the next K-tile are read while this one's
// MFMAs run, plane by plane as a plane's last MFMA has been issued (x1 y1, x1 y0, x0 y1, then plane 2's, x0 y0 last). So one
// register set holds each plane, and the barrier stands behind x1 y1, under which plane 0 arrives. 238 registers for a wavefront
// of 64 x 64 with both accumulators, none spilled. The operands are passed (B, A): a lane then holds four neighbouring columns
// of one row of C, stored as one vector. Persistent: workgroups walk the tiles `grid` apart, loads run ahead across tile borders.
// Bound by the matrix units and the power they draw: 4096^3 264 TFLOP/s of fp32 products, 1.58 PFLOP/s of bf16 ones (fp32 MFMA
// kernel: 146); by counter the matrix units are busy in 0.74 of the cycles at a clock of 1.7 GHz (nominal 2.4), without an LDS
// bank conflict.
template <int BM, int BN, int WM, int WN, bool ROWMAX>
__global__ __launch_bounds__(WM *WN *kWave, 2) void plane_gemm_kernel(const PlaneArgs p) {
    constexpr int NW = WM * WN;
    constexpr int WTM = BM / WM, WTN = BN / WN, TM = WTM / 16, TN = WTN / 16;
    constexpr int BUF = kPlanes * (BM + BN) * 64;                          // bytes: A planes [3][BM][64], then B planes [3][BN][64]
    constexpr int A_CH = kPlanes * BM / 16, B_CH = kPlanes * BN / 16;      // 1 KB blocks of a K-tile
    constexpr int LA = (A_CH + NW - 1) / NW, LB = (B_CH + NW - 1) / NW;
    static_assert(!ROWMAX || WTN == 64, "row maxima are kept per 64 columns");
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm0 = (wave / WN) * WTM, wn0 = (wave % WN) * WTN;
    const int l16 = lane & 15, lq = lane >> 4;
    const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)reinterpret_cast<uintptr_t>(smem));
    const int grid = (int)gridDim.x;
    const int vb = xcd_contiguous_id((int)blockIdx.x, grid);
    const int items = p.tiles * p.splits;
    if (vb >= items) return;

    auto run_of = [&](int item, int &first) __attribute__((always_inline)) {
        const int s = item / p.tiles;
        first = s * p.kt_per;
        const int rest = p.ktiles - first;
        return rest < p.kt_per ? rest : p.kt_per;
    };
    // ---- loader: one K-tile ahead of the operand reads ----
    int ld_item = vb;
    int ld_left = 0;  // K-tiles of ld_item still to request
    const unsigned char *ak = nullptr, *bk = nullptr;
    unsigned a_off[LA], b_off[LB];  // byte offsets of this wavefront's blocks (uniform)
    const int64_t a_step = (int64_t)p.a_blocks * kPlanes * kBlock, b_step = (int64_t)p.b_blocks * kPlanes * kBlock;
    auto setup = [&]() __attribute__((always_inline)) {
        int tm, tn, first;
        ld_left = __builtin_amdgcn_readfirstlane(run_of(ld_item, first));
        tile_of_id(ld_item % p.tiles, p.tiles_m, p.tiles_n, p.order, tm, tn);
        ak = uniform_ptr(p.a + first * a_step);
        bk = uniform_ptr(p.b + first * b_step);
#pragma unroll
        for (int i = 0; i < LA; ++i) {
            const int c = i * NW + wave;
            int blk = tm * (BM / 16) + c % (BM / 16);
            blk = blk < p.a_blocks ? blk : p.a_blocks - 1;
            a_off[i] = __builtin_amdgcn_readfirstlane((unsigned)(c / (BM / 16) * p.a_blocks + blk) * (unsigned)kBlock);
        }
#pragma unroll
        for (int i = 0; i < LB; ++i) {
            const int c = i * NW + wave;
            int blk = tn * (BN / 16) + c % (BN / 16);
            blk = blk < p.b_blocks ? blk : p.b_blocks - 1;
            b_off[i] = __builtin_amdgcn_readfirstlane((unsigned)(c / (BN / 16) * p.b_blocks + blk) * (unsigned)kBlock);
        }
    };
    const unsigned wdst = lds0 + (unsigned)wave * kBlock;
    auto issue = [&](int buf) __attribute__((always_inline)) {
        if (ld_left == 0) return;  // past the last K-tile of this workgroup
#pragma unroll
        for (int i = 0; i < LA; ++i)
            if (A_CH % NW == 0 || i + 1 < LA || i * NW + wave < A_CH) load_to_lds_16(ak + a_off[i], lane * 16u, wdst + buf * BUF + i * NW * kBlock);
#pragma unroll
        for (int i = 0; i < LB; ++i)
            if (B_CH % NW == 0 || i + 1 < LB || i * NW + wave < B_CH) load_to_lds_16(bk + b_off[i], lane * 16u, wdst + buf * BUF + (A_CH + i * NW) * kBlock);
        ak += a_step;
        bk += b_step;
        if (--ld_left == 0) {
            ld_item += grid;
            if (ld_item < items) setup();
        }
    };

    struct Frag { bf16x8 a[TM], b[TN]; };
    const int a_rd = (wm0 + l16) * 64 + ((lq ^ fth::swz(l16)) << 4), b_rd = A_CH * kBlock + (wn0 + l16) * 64 + ((lq ^ fth::swz(l16)) << 4);
    auto fetch = [&](Frag &f, int buf, int s) __attribute__((always_inline)) {
        const unsigned char *s0 = smem + buf * BUF;
#pragma unroll
        for (int i = 0; i < TM; ++i) f.a[i] = *reinterpret_cast<const bf16x8 *>(s0 + s * BM * 64 + a_rd + i * kBlock);
#pragma unroll
        for (int j = 0; j < TN; ++j) f.b[j] = *reinterpret_cast<const bf16x8 *>(s0 + s * BN * 64 + b_rd + j * kBlock);
    };
    f32x4 acc[TM][TN], low[TM][TN];  // sums of x0 y0, and of the five products with a lower part
    auto mul = [&](f32x4 (&to)[TM][TN], const Frag &fa, const Frag &fb) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) to[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb.b[j], fa.a[i], to[i][j], 0, 0, 0);
    };
    auto zero = [&](f32x4 (&to)[TM][TN]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) to[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    };

    // This wavefront's part of a tile again, from the fp32 operands. us, fp32 kernels / here with one NaN in A / with every sum
    // computed again: 4096^3 935 / 930 / 1690, 8192 x 3072 x 768 284 / 234 / 481, 2331 x 768 x 768 40 / 74 / 72 (a tile's second
    // pass is a chain of its own K on one wavefront).
    auto again = [&](int64_t m0, int64_t n0, int first, int nk, int l16, int lq) __attribute__((always_inline)) {
        zero(acc);
        const fth::SplitGemm &g = p.g;
        const int k_first = first * kBK + lq * 4;
        int left = (int)((first + nk) * kBK < g.k ? (first + nk) * kBK : g.k) - k_first;  // k of this lane's row pieces still to load
        const float *pa[TM], *pb[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int64_t row = m0 + i * 16 + l16;
            pa[i] = g.a + (row < g.m ? row : g.m - 1) * g.a_rs + k_first * g.a_ks;
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int64_t col = n0 + j * 16 + l16;
            pb[j] = g.b + (col < g.n ? col : g.n - 1) * g.b_rs + k_first * g.b_ks;
        }
        f32x4 av[TM], bv[TN];
        auto load = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                av[i] = four_k(pa[i], g.a_ks, left);
                pa[i] += 16 * g.a_ks;
            }
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                bv[j] = four_k(pb[j], g.b_ks, left);
                pb[j] += 16 * g.b_ks;
            }
            left -= 16;
        };
        load();
        for (int it = 0; it < 2 * nk; ++it) {  // 16 k at a time, the next ones requested ahead of this one's MFMAs
            f32x4 ma[TM], mb[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i) ma[i] = av[i];
#pragma unroll
            for (int j = 0; j < TN; ++j) mb[j] = bv[j];
            load();
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(mb[j][e], ma[i][e], acc[i][j], 0, 0, 0);
        }
    };

    auto finish = [&](int item, int first, int nk) __attribute__((always_inline)) {
        int at = lane;
        asm volatile("" : "+v"(at));  // nothing of the output's addresses is worked out ahead of the loop and held through it
        const int l16 = at & 15, lq = at >> 4;
        int tm, tn;
        tile_of_id(item % p.tiles, p.tiles_m, p.tiles_n, p.order, tm, tn);
        const int64_t m0 = (int64_t)tm * BM + wm0, n0 = (int64_t)tn * BN + wn0;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] += low[i][j];
        float big = 0.f, small = FLT_MAX;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    big = nan_max(big, __builtin_fabsf(acc[i][j][e]));
                    small = __builtin_fminf(small, __builtin_fabsf(acc[i][j][e]));
                }
        if (__builtin_amdgcn_ballot_w64(!(big <= FLT_MAX) || small < kTiny)) {  // rare: look closer (exact zeros are exact)
            bool doubt = !(big <= FLT_MAX);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) doubt = doubt || (acc[i][j][e] != 0.f && __builtin_fabsf(acc[i][j][e]) < kTiny);
            if (__builtin_amdgcn_ballot_w64(doubt)) again(m0, n0, first, nk, l16, lq);
        }
        const int64_t m = p.g.m, n = p.g.n;
        const bool parts = p.splits > 1;
        float *c = parts ? p.partial + (int64_t)(item / p.tiles) * m * n : p.g.c;
        const int64_t ldc = parts ? n : p.g.ldc;
        if (!parts) {
            if (p.g.alpha != 1.f) {
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j) acc[i][j] *= p.g.alpha;
            }
            if (p.g.epilogue & FTH_EPI_BIAS) {
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int64_t col = n0 + j * 16 + lq * 4 + e;
                        const float b = col < n ? p.g.bias[col] : 0.f;
#pragma unroll
                        for (int i = 0; i < TM; ++i) acc[i][j][e] += b;
                    }
            }
            if (p.g.epilogue & FTH_EPI_GELU) {
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[i][j][e] = fth::gelu_erf(acc[i][j][e]);
            } else if (p.g.epilogue & FTH_EPI_GELU_TANH) {
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[i][j][e] = fth::gelu_tanh(acc[i][j][e]);
            }
        }
        const float *res = !parts && (p.g.epilogue & FTH_EPI_RESIDUAL) ? p.g.residual : nullptr;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int64_t row = m0 + i * 16 + l16;
            float top = -__builtin_inff();
            if (row < m) {
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    const int64_t col = n0 + j * 16 + lq * 4;
                    float *dst = c + row * ldc + col;
                    if (col + 4 <= n) {
                        if (res) acc[i][j] += *reinterpret_cast<const f32x4_any *>(res + row * ldc + col);
                        *reinterpret_cast<f32x4_any *>(dst) = acc[i][j];
                        if constexpr (ROWMAX)
#pragma unroll
                            for (int e = 0; e < 4; ++e) top = nan_max(top, acc[i][j][e]);
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (col + e < n) {
                                const float v = res ? acc[i][j][e] + res[row * ldc + col + e] : acc[i][j][e];
                                dst[e] = v;
                                if constexpr (ROWMAX) top = nan_max(top, v);
                            }
                    }
                }
            }
            if constexpr (ROWMAX) {
                top = nan_max(top, __shfl_xor(top, 16));
                top = nan_max(top, __shfl_xor(top, 32));
                const int64_t group = n0 / 64;
                if (lq == 0 && row < m && group < p.rowmax_groups) p.g.rowmax[group * m + row] = top;
            }
        }
    };

    Frag f0, f1, f2;  // this K-tile's operands by plane
    auto fetch_all = [&](int buf) __attribute__((always_inline)) {
        fetch(f1, buf, 1);
        fetch(f0, buf, 0);
        fetch(f2, buf, 2);
    };
    // One K-tile. The next K-tile's own loads have landed behind the wait, everyone's behind the barrier, and everyone has this
    // K-tile's operands in registers. After the last K-tile of a tile the reads fetch what is left there.
    auto step = [&](int buf) __attribute__((always_inline)) {
        mul(low, f1, f1);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0x0F70);
        __syncthreads();
        issue(buf);
        mul(low, f1, f0);
        mul(low, f0, f1);
        __builtin_amdgcn_sched_barrier(0);
        fetch(f1, buf ^ 1, 1);
        mul(low, f2, f0);
        mul(low, f0, f2);
        __builtin_amdgcn_sched_barrier(0);
        fetch(f2, buf ^ 1, 2);
        mul(acc, f0, f0);
        __builtin_amdgcn_sched_barrier(0);
        fetch(f0, buf ^ 1, 0);
    };
    int buf = 0;
    setup();
    issue(0);
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): own part landed
    __syncthreads();
    issue(1);
    for (int item = vb; item < items; item += grid) {
        int first;
        const int nk = __builtin_amdgcn_readfirstlane(run_of(item, first));
        zero(acc);
        zero(low);
        fetch_all(buf);  // (nothing of the next tile is held in registers across the output)
        for (int kt = 0; kt < nk; ++kt) {
            step(buf);
            buf ^= 1;
        }
        finish(item, first, nk);
    }
}

// Sum of the split runs in K order, then the epilogue.
__global__ __launch_bounds__(256) void plane_reduce_kernel(const PlaneArgs p) {
    const int64_t n = p.g.n, total = p.g.m * n;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    float v = p.partial[i];
    for (int s = 1; s < p.splits; ++s) v += p.partial[s * total + i];
    const int64_t row = i / n, col = i - row * n;
    if (p.g.alpha != 1.f) v *= p.g.alpha;
    if (p.g.epilogue & FTH_EPI_BIAS) v += p.g.bias[col];
    if (p.g.epilogue & FTH_EPI_GELU) v = fth::gelu_erf(v);
    if (p.g.epilogue & FTH_EPI_GELU_TANH) v = fth::gelu_tanh(v);
    if (p.g.epilogue & FTH_EPI_RESIDUAL) v += p.g.residual[row * p.g.ldc + col];
    p.g.c[row * p.g.ldc + col] = v;
}

// ---- which tile, how many runs of K ----

// One workgroup of 128 x 256, 128 x 192 or 128 x 128 a compute unit, or two of 64 x 128. Rates are TFLOP/s of fp32 products with every
// compute unit busy, measured on 4096^3, 8192 x 768 x 3072, 4662 x 768 x 768 and 2331 x 768 x 768; the small tile's with one and with
// two workgroups on a compute unit, the others' in one round and in more. The square tile gains most where it makes one round and the
// small one two; in full rounds it is behind the wide one (4096^3 614 us, 581), and of several rounds it is taken where its last one
// comes out fuller (us without / with it: 20011 x 1000 x 520 151 / 148, 1224 x 15221 x 1768 391 / 381, 8239 x 2886 x 600 180 / 173): 1031 x 3072
// x 768 42.9 -> 39.2 us, planes included, 3000 x 1024 x 1024 52.0 -> 47.4, 4662 x 768 x 768 44.5 -> 42.3, 6000 x 512 x 512 35.3 -> 33.7.
struct Tile { int bm, bn; double rate[2]; };
constexpr Tile kTiles[] = {{128, 256, {250., 250.}}, {128, 192, {238., 238.}}, {64, 128, {145., 200.}}, {128, 128, {255., 225.}}};
constexpr int kResident[] = {1, 1, 2, 1};

struct Choice { int tile = -1, splits = 1, kt_per = 0; double us = 0; };

// Time of the product alone: the tiles that the busiest compute unit works through, and for split K the partial sums' way
// through memory (written and read at 4 TB/s, 4 us for the second launch).
Choice choose(int64_t m, int64_t n, int64_t k, bool rowmax) {
    const int cus = fth::compute_units() > 0 ? fth::compute_units() : 256;
    const int64_t ktiles = fth::ceil_div(k, kBK);
    Choice best;
    for (int t = 0; t < (rowmax ? 1 : 4); ++t) {
        const Tile &c = kTiles[t];
        const int64_t tiles = fth::ceil_div(m, c.bm) * fth::ceil_div(n, c.bn);
        for (int s = 1; s <= (rowmax || t == 3 ? 1 : 16); ++s) {  // (the square tile with a split K: 5246 x 320 x 896 43 us, 40 without it)
            const int64_t per = fth::ceil_div(ktiles, s);
            if (s > 1 && (per < 8 || (s - 1) * per >= ktiles)) break;
            const int64_t most = fth::ceil_div(tiles * s, (int64_t)cus);
            const double one = 2.0 * c.bm * c.bn * kBK * per * cus * 1e-6;
            double us = 2.0 + 2.0 * most / kResident[t];
            us += kResident[t] == 1 ? most * one / c.rate[most > 1] : (most / 2) * 2 * one / c.rate[1] + (most % 2) * one / c.rate[0];
            if (s > 1) us += (s + 1.0) * m * n * 4 / 4e6 + 4.0;
            if (best.tile < 0 || us < best.us) best = {t, s, (int)per, us};
        }
    }
    return best;
}

size_t plane_bytes(int64_t rows, int64_t k) { return (size_t)(fth::ceil_div(k, kBK) * kPlanes * fth::ceil_div(rows, 16)) * kBlock; }

template <int BM, int BN, int WM, int WN, bool ROWMAX> int32_t launch_planes(PlaneArgs &p, int per_cu, hipStream_t st) {
    constexpr int smem = 2 * kPlanes * (BM + BN) * 64;
    auto kern = plane_gemm_kernel<BM, BN, WM, WN, ROWMAX>;
    static const hipError_t ready = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    FTH_HIP(ready);
    p.tiles_m = (int)fth::ceil_div(p.g.m, BM);
    p.tiles_n = (int)fth::ceil_div(p.g.n, BN);
    p.tiles = p.tiles_m * p.tiles_n;  // (m n is at most 2^31)
    p.order = p.tiles_n > p.tiles_m ? 1 : 0;
    const int64_t slots = (int64_t)(fth::compute_units() > 0 ? fth::compute_units() : 256) * per_cu, items = p.tiles * p.splits;
    kern<<<dim3((unsigned)(items < slots ? items : slots)), dim3(WM * WN * kWave), smem, st>>>(p);
    FTH_CHECK_LAUNCH("gemm_planes");
    return FTH_OK;
}

SplitArgs split_args(const float *x, unsigned char *planes, int64_t rows, int64_t k, int64_t rs, int64_t ks) {
    SplitArgs o{x, planes, rows, k, ks == 1 ? rs : ks, (int)fth::ceil_div(rows, 16), (int)fth::ceil_div(k, kBK), ks == 1, 0};
    o.groups = o.by_k ? fth::ceil_div(o.ktiles, 4) * o.blocks : fth::ceil_div(o.blocks, 4) * o.ktiles;
    return o;
}

int32_t run_split(const fth::SplitGemm &g, const Choice &ch, unsigned char *scratch, hipStream_t st) {
    PlaneArgs p{};
    p.g = g;
    p.ktiles = (int)fth::ceil_div(g.k, kBK);
    p.a_blocks = (int)fth::ceil_div(g.m, 16);
    p.b_blocks = (int)fth::ceil_div(g.n, 16);
    p.splits = ch.splits;
    p.kt_per = ch.kt_per;
    p.rowmax_groups = fth::gemm_rowmax_groups(g.n);
    unsigned char *pa = scratch, *pb = pa + plane_bytes(g.m, g.k);
    p.a = pa;
    p.b = pb;
    p.partial = reinterpret_cast<float *>(pb + plane_bytes(g.n, g.k));
    const SplitArgs sa = split_args(g.a, pa, g.m, g.k, g.a_rs, g.a_ks), sb = split_args(g.b, pb, g.n, g.k, g.b_rs, g.b_ks);
    split_kernel<<<dim3((unsigned)(sa.groups + sb.groups)), dim3(256), 0, st>>>(sa, sb);
    FTH_CHECK_LAUNCH("gemm_split");
    int32_t rc = FTH_OK;
    switch (ch.tile) {
        case 0:
            rc = g.rowmax ? launch_planes<128, 256, 2, 4, true>(p, kResident[0], st) : launch_planes<128, 256, 2, 4, false>(p, kResident[0], st);
            break;
        case 1: rc = launch_planes<128, 192, 2, 4, false>(p, kResident[1], st); break;
        case 2: rc = launch_planes<64, 128, 2, 2, false>(p, kResident[2], st); break;
        default: rc = launch_planes<128, 128, 2, 4, false>(p, kResident[3], st); break;
    }
    if (rc || ch.splits == 1) return rc;
    plane_reduce_kernel<<<dim3((unsigned)fth::ceil_div(g.m * g.n, 256)), dim3(256), 0, st>>>(p);
    FTH_CHECK_LAUNCH("gemm_planes_reduce");
    return FTH_OK;
}

size_t scratch_bytes(int64_t m, int64_t n, int64_t k, const Choice &ch) {
    return plane_bytes(m, k) + plane_bytes(n, k) + (ch.splits > 1 ? (size_t)ch.splits * m * n * sizeof(float) : 0);
}

}  // namespace

namespace fth {

bool split_gemm_pays(const SplitGemm &g, SplitRival rival) {
    static const bool off = [] {
        const char *e = std::getenv("FT_HIP_GEMM_SPLIT");  // tuning knob: 0 keeps large products on fp32 MFMAs
        return e && std::atoi(e) == 0;
    }();
    // Under 1.5 GFLOP the fp32 path has its own small kernels and the launches decide: a 128 x 256 x 256 block would lose 26 us.
    const int64_t m = g.m, n = g.n, k = g.k;
    const double flop = 2.0 * m * n * k;
    if (off || m < 64 || n < 64 || k < 128 || flop < 1.5e9 || m > (1 << 20) || n > (1 << 20) || k > (1 << 20) || m * n > ((int64_t)1 << 31)) return false;
    const Choice ch = choose(m, n, k, g.rowmax != nullptr);
    if (scratch_bytes(m, n, k, ch) > kStreamScratchMost) return false;
    // This path: the product, the planes at 10 bytes an element (12 where it is stored [k][rows]), 4.5 TB/s and 3 us, and for less
    // than 256 k the output's way to memory. The fp32 kernels: 130 TFLOP/s and 16 us (whole-tile effects and the fix-up pass of a
    // split K) with direct-to-LDS operands, but 7 us where 128 x 96 tiles come out even; 0.69 of that rate and 25 us with 128-bit
    // loads, 0.59 and 16 us with single ones; the transposed copy of a ragged [k, m] operand. The second is the least certain of the three. us, fp32 -> split: 2331 x 768 x 768
    // 44 -> 32, 768 x 768 x 2331 (A stored [k, m]) 62 -> 38, 4000 x 1024 x 1024 83 -> 55, 1414 x 2504 x 224 35 -> 23; near the line,
    // 303 x 10360 x 288 35 -> 31, 360 x 528 x 4304 38 -> 32, 256 x 816 x 4479 46 -> 34; past it, 8192 x 768 x 128 20 -> 22, with B
    // stored [k, n] 198 x 6752 x 7868 241 -> 265 and 256 x 5704 x 7844 209 -> 226.
    const int64_t slots = 2 * (int64_t)(compute_units() > 0 ? compute_units() : 256);
    const bool even = rival == SplitRival::Direct && g.a_ks == 1 && n % 96 == 0 && ceil_div(m, 128) * (n / 96) % slots == 0 &&
                      ceil_div(m, 128) * ceil_div(n, 128) % slots != 0;  // (as the fp32 path chooses them)
    const double out_us = k < 256 ? 4.0 * m * n / 6.5e6 : 0.0;
    const double planes_us = ((g.a_ks == 1 ? 10.0 : 12.0) * m + (g.b_ks == 1 ? 10.0 : 12.0) * n) * k / 4.5e6 + 3.0;
    const double ours = ch.us + planes_us + out_us, copy_us = g.a_ks == 1 ? 0.0 : 8.0 * m * k / 4.5e6;
    switch (rival) {
        case SplitRival::Direct: return ours < 0.95 * (flop / 130e6 + (even ? 7.0 : 16.0 + out_us));
        case SplitRival::Copied: return ours < 1.08 * (flop / 130e6 + 16.0 + out_us + copy_us);
        case SplitRival::Vector: return ours < 0.85 * (flop / (0.69 * 130e6) + 25.0 + out_us + copy_us);
        default: return ours < 1.02 * (flop / (0.59 * 130e6) + 16.0 + out_us);
    }
}

bool split_gemm(const SplitGemm &g, hipStream_t st, int32_t *rc) {
    const Choice ch = choose(g.m, g.n, g.k, g.rowmax != nullptr);
    StreamScratch lease;
    void *scratch = lease.get(st, ScratchUse::SplitPlanes, scratch_bytes(g.m, g.n, g.k, ch));
    if (!scratch) return false;
    *rc = run_split(g, ch, static_cast<unsigned char *>(scratch), st);
    return true;
}

}  // namespace fth
