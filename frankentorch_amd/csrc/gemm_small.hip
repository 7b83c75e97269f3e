// fp32 products of few rows, or of little work (the 128-token transformer block: 17 to 67 MFLOP a product; a decoder's products
// for a few tokens, which read every weight for little arithmetic).
//
// One launch, no fix-up pass: a workgroup owns MT x NT output tiles of 16 x 16 and splits K over its NW wavefronts, which feed
// v_mfma_f32_16x16x4_f32 from memory without a barrier; the NW partial tiles are added through LDS in wavefront order, so the sum
// order is fixed by the shape.
//
// Bound by the path into a compute unit. A wavefront's 128-bit load reaches 64 bytes a cycle when four neighbouring lanes
// read 64 neighbouring bytes, and a quarter of that when neighbouring lanes read different rows, which is what the MFMA's operand
// layout asks for (measured from L2: 149 against 38 KB/us a compute unit). So a wavefront loads 16 rows x 64 bytes with four lanes a
// row and turns the kilobyte into the operand layout through LDS of its own: a write, a read, no barrier (a wavefront's LDS
// instructions execute in order). U such loads of each operand are in flight, and a slot is requested again as soon as it is
// used, so weights that come from HBM pay its latency once.
// The MFMAs of one pass over the U loads (chains of 16 or 24; of 8 with two slots) are added to a sum with ordinary additions before the
// next pass, so that a long K does not grow the error with its root: a chain of L MFMAs loses 5e-8 sqrt(L / 2). Relative 2-norm
// error against 64 bits, kernels before (K cut over more wavefronts or workgroups) / one chain a wavefront / here: 37 x 2304 x 768 1.9e-7 / 2.5e-7 /
// 1.5e-7, 200 x 1536 x 512 1.55e-7 / 2.1e-7 / 1.5e-7, 64 x 5000 x 992 2.1e-7 / 2.9e-7 / 1.6e-7, 64 x 512 x 16384 2.9e-7 / 8.1e-7 / 1.9e-7; us without and
// with the sums 5.27 / 5.42, 7.34 / 7.30, 11.6 / 11.6, 30.2 / 30.5, 400 x 2304 x 768 21.4 / 22.1.

#include <cstdlib>

#include "devmath.hpp"
#include "gemm_small.hpp"

namespace {

constexpr int kXcds = 8;

using Acc4 = __attribute__((ext_vector_type(4))) float;

template <int NW, int MT, int NT, int U, bool TRANS_B>
__global__ __launch_bounds__(64 * NW) void gemm_quad_kernel(const fth::SmallGemm p, const int tiles_m, const int tiles_n) {
    constexpr int TILE = 1024, SLOT = (MT + (TRANS_B ? NT : 0)) * TILE;  // 16 rows x 64 bytes; what a group of 16 k takes
    constexpr int PITCH = 17;
    static_assert(TRANS_B || NT == 1, "several column tiles share the rows of A that went through LDS");
    constexpr int PART = MT * NT * 16 * PITCH * 4;  // a wavefront's partial tiles reuse its staging area
    constexpr int AREA = 2 * SLOT > PART ? 2 * SLOT : PART;
    __shared__ __attribute__((aligned(16))) unsigned char smem[NW][AREA];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lrow = lane & 15, g = lane >> 4;  // operand layout: row, and which four of 16 k
    const int qrow = lane >> 2, qc = lane & 3;  // load layout
    // The row tiles of one column tile are eight workgroups apart: on one XCD, whose L2 then reads B's rows from memory once.
    const int run = kXcds * tiles_m, first_n = (int)blockIdx.x / run * kXcds, in_run = (int)blockIdx.x % run;
    const int width = tiles_n - first_n < kXcds ? tiles_n - first_n : kXcds;
    const int tile_m = in_run / width, tile_n = first_n + in_run % width;
    const int64_t batch = blockIdx.y, m0 = (int64_t)tile_m * (16 * MT), n0 = (int64_t)tile_n * (16 * NT);
    // this wavefront's K range: whole groups of 16, contiguous, in wavefront order
    const int groups = (int)(p.k / 16), per = (groups + NW - 1) / NW;
    const int g0 = wave * per, g1 = g0 + per < groups ? g0 + per : groups, last = groups - 1;
    const float *A = p.a + batch * p.stride_a, *B = p.b + batch * p.stride_b;
    const float *ap[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {  // rows past the edge read the last valid row; they are never stored
        const int64_t row = m0 + i * 16 + qrow;
        ap[i] = A + (row < p.m ? row : p.m - 1) * p.lda + 4 * qc;
    }
    const float *bp[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        int64_t br = n0 + j * 16 + (TRANS_B ? qrow : lrow);
        br = br < p.n ? br : p.n - 1;
        bp[j] = TRANS_B ? B + br * p.ldb + 4 * qc : B + (int64_t)(4 * g) * p.ldb + br;
    }

    Acc4 av[U][MT], bv[U][NT];
    auto load = [&](int u, int group) __attribute__((always_inline)) {
        const int t = group < last ? group : last;
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            if (TRANS_B) {
                bv[u][j] = *reinterpret_cast<const Acc4 *>(bp[j] + 16 * t);
            } else {
                const float *bk = bp[j] + (int64_t)(16 * t) * p.ldb;
                bv[u][j] = Acc4{bk[0], bk[p.ldb], bk[2 * p.ldb], bk[3 * p.ldb]};
            }
        }
#pragma unroll
        for (int i = 0; i < MT; ++i) av[u][i] = *reinterpret_cast<const Acc4 *>(ap[i] + 16 * t);
    };
    unsigned char *area = smem[wave];
    const int wr = qrow * 64 + ((qc ^ fth::swz(qrow)) << 4), rd = lrow * 64 + ((g ^ fth::swz(lrow)) << 4);
    Acc4 sum[MT][NT], acc[MT][NT];
    auto clear = [](Acc4 (&x)[MT][NT]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) x[i][j] = Acc4{0.f, 0.f, 0.f, 0.f};
    };
    auto collect = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) sum[i][j] += acc[i][j];
    };
    clear(sum);
    auto stage = [&](int u) __attribute__((always_inline)) {
        unsigned char *s = area + (u & 1) * SLOT + wr;
#pragma unroll
        for (int i = 0; i < MT; ++i) *reinterpret_cast<Acc4 *>(s + i * TILE) = av[u][i];
        if (TRANS_B)
#pragma unroll
            for (int j = 0; j < NT; ++j) *reinterpret_cast<Acc4 *>(s + (MT + j) * TILE) = bv[u][j];
    };
    auto multiply = [&](int u, const Acc4 (&direct)[NT]) __attribute__((always_inline)) {
        const unsigned char *s = area + (u & 1) * SLOT + rd;
        Acc4 b[NT];
#pragma unroll
        for (int j = 0; j < NT; ++j) b[j] = TRANS_B ? *reinterpret_cast<const Acc4 *>(s + (MT + j) * TILE) : direct[j];
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const Acc4 a = *reinterpret_cast<const Acc4 *>(s + i * TILE);
            // step e contracts k = 16 t + 4 g + e over the four lane groups
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[j][e], acc[i][j], 0, 0, 0);
        }
    };
#pragma unroll
    for (int u = 0; u < U; ++u) load(u, g0 + u);
    int t0 = g0;
    for (; t0 + U < g1; t0 += U) {
        clear(acc);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            stage(u);
            Acc4 b[NT];
#pragma unroll
            for (int j = 0; j < NT; ++j) b[j] = bv[u][j];
            load(u, t0 + U + u);
            multiply(u, b);
        }
        collect();
    }
    clear(acc);
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (t0 + u < g1) {
            stage(u);
            multiply(u, bv[u]);
        }
    collect();
    float *part = reinterpret_cast<float *>(area);  // (this wavefront's reads of it are done: LDS instructions execute in order)
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) part[((i * NT + j) * 16 + 4 * g + r) * PITCH + lrow] = sum[i][j][r];  // accumulator element r: row 4 g + r, column lrow
    __syncthreads();
    float *C = p.c + batch * p.stride_c;
#pragma unroll
    for (int e = tid; e < MT * NT * 256; e += 64 * NW) {
        const int c = e % (16 * NT), r = e / (16 * NT);
        const int64_t row = m0 + r, col = n0 + c;
        if (row < p.m && col < p.n) {
            const float *first = reinterpret_cast<const float *>(smem[0]) + ((r / 16 * NT + c / 16) * 16 + r % 16) * PITCH + c % 16;
            float v = *first;
#pragma unroll
            for (int w = 1; w < NW; ++w) v += first[w * (AREA / 4)];
            if (p.alpha != 1.f) v = p.alpha * v;
            if (p.epilogue & FTH_EPI_BIAS) v = v + p.bias[col];
            if (p.epilogue & FTH_EPI_GELU) v = fth::gelu_erf(v);
            if (p.epilogue & FTH_EPI_GELU_TANH) v = fth::gelu_tanh(v);
            if (p.epilogue & FTH_EPI_RESIDUAL) v = v + p.residual[batch * p.stride_c + row * p.ldc + col];
            C[row * p.ldc + col] = v;
        }
    }
}

template <int NW, int MT, int NT, int U, bool TRANS_B> int32_t launch(const fth::SmallGemm &g, hipStream_t st) {
    const int tiles_m = (int)fth::ceil_div(g.m, 16 * MT), tiles_n = (int)fth::ceil_div(g.n, 16 * NT);
    gemm_quad_kernel<NW, MT, NT, U, TRANS_B><<<dim3((unsigned)(tiles_m * tiles_n), (unsigned)g.batch), dim3(64 * NW), 0, st>>>(g, tiles_m, tiles_n);
    FTH_CHECK_LAUNCH("gemm_small");
    return FTH_OK;
}

// Which form. Few tiles, or long reductions but for very many: eight wavefronts; otherwise four, whose partial tiles are less to add up; two row tiles
// a workgroup, then two column tiles as well, once there are workgroups enough: rows of A come from L2 less often. Six slots where they come out even (K 768 and 3072 over eight wavefronts).
// us, eight wavefronts / four / four with two row tiles: 37 x 768 x 3072 9.2 / 13.6 / -, 37 x 2304 x 768 6.4 / 6.3 / 8.1, 200 x 1536 x 512
// 8.2 / 7.0 / 7.8, 9 x 3072 x 768 5.1 / 5.7 / -, 64 x 50257 x 768 - / 87 / 79; with 2 x 2 tiles 65, 37 x 50257 x 768 58.6, with 3 x 2 55.6
// (2 x 1: 62.3; 33 to 48 rows with 2 x 2 / 3 x 2, weights mostly from HBM: 33 x 33009 x 272 20.7 / 18.4, 41 x 32000 x 1024 54 / 46, 36 x 100000 x 256
// 49 / 38, 33 x 32768 x 2048 99 / 82, 48 x 128256 x 1024 206 / 185, 41 x 25000 x 4096 180 / 175), 400 x 2304 x 768 20.2 (21.8); 64 x 10000 x 768 16.4 (16.1). 64 x 32000 x 1024
// eight wavefronts 75, four with 2 x 2 tiles 52.
template <bool TRANS_B> int32_t choose(const fth::SmallGemm &g, hipStream_t st) {
    const int64_t tiles = fth::ceil_div(g.m, 16) * fth::ceil_div(g.n, 16) * g.batch, per = fth::ceil_div(g.k / 16, 8);
    if (tiles <= 288 || (g.k >= 1024 && tiles < 1536)) return per % 6 == 0 ? launch<8, 1, 1, 6, TRANS_B>(g, st) : launch<8, 1, 1, 4, TRANS_B>(g, st);
    if (tiles < 1536 || g.m <= 16) return launch<4, 1, 1, 4, TRANS_B>(g, st);
    if constexpr (TRANS_B) {
        if (tiles >= 6000 && g.m > 32 && g.m <= 48) return launch<4, 3, 2, 2, true>(g, st);
        if (tiles >= 3072) return launch<4, 2, 2, 2, true>(g, st);
    }
    return launch<4, 2, 1, 4, TRANS_B>(g, st);
}

}  // namespace

namespace fth {

bool small_gemm(const SmallGemm &g, hipStream_t st, int32_t *rc) {
    static const bool off = [] {
        const char *e = std::getenv("FT_HIP_GEMM_SMALL");  // tuning knob: 0 sends small problems to the large-tile kernels
        return e && std::atoi(e) == 0;
    }();
    const double flop = 2.0 * (double)g.m * (double)g.n * (double)g.k * (double)g.batch;
    const int64_t tiles = ceil_div(g.m, 16) * ceil_div(g.n, 16);
    if (off || g.k % 16 != 0 || g.batch > 65535 || tiles > (1 << 24)) return false;
    // Where it is the fastest, us of the kernels behind it / here, from a sweep of 21 (n, k) pairs and 18 m, both forms of B:
    // [n, k] B: K of 256 and more (2048 x 1000 x 64 8.3 / 11.6, 333 x 8192 x 128 13.3 / 17.9, but 1024 x 768 x 256 15.6 / 8.9). Up to 64
    // rows at any size (64 x 50257 x 768 97 / 65, 48 x 4096 x 4096 38 / 31). More rows: under 1.5 GFLOP, where the split product begins
    // (400 x 2304 x 768 28.8 / 20.9, 1600 x 1152 x 384 31.5 / 21.9), and around K 768 up to 2 GFLOP where that one is not taken (1600 x 768 x 768 33.2 / 27.5, 128 x
    // 10000 x 768 34.7 / 29.4; not 2048 x 768 x 768 36.7 / 43.2, 1300 x 1536 x 512 25.7 / 27.7, 1300 x 384 x 1536 29.6 / 31.3).
    // The longest K belong to the kernels that cut K over many workgroups, which these few tiles leave idle: 64 x 128 x 131072 192 / 217,
    // 16 x 256 x 131072 187 / 216; but 64 x 128 x 98304 189 / 145, 64 x 64 x 100000 270 / 164, 64 x 512 x 65536 130 / 109, 128 x 128 x 40000
    // 111 / 73, 64 x 4096 x 11008 105 / 85, and where there is too little work for them 1 x 128 x 262144 830 / 420, 64 x 32 x 200000 352 / 337.
    // Batches: 64 x 64 x 4096, 32 of them 35 / 31, 64 x 256 x 16384, eight 88 / 75, 64 x 128 x 256, 200 of them 22.5 / 19.2.
    // [k, n] B, whose loads are in the MFMA layout to begin with: mid-sized products (400 x 2304 x 768 28.5 / 23.8, 1600 x 1152 x 384
    // 31.4 / 24.1; not 24 x 2304 x 768 5.75 / 6.6, 777 x 512 x 2048 30.1 / 37.3).
    if (g.trans_b) {
        if (g.k < 256 || (g.m > 64 && flop >= (g.k >= 640 && g.k <= 1024 ? 2.0e9 : 1.5e9)) || (g.k > 114688 && flop > 1.0e9)) return false;
    } else if (g.k < 384 || g.k > 1536 || flop < 1.0e8 || flop >= 1.5e9) {
        return false;
    }
    *rc = g.trans_b ? choose<true>(g, st) : choose<false>(g, st);
    return true;
}

}  // namespace fth
