// float64 products of middling size, on v_mfma_f64_16x16x4_f64, in one launch.
//
// A workgroup owns a 32 x 32 output tile and splits K over its NW wavefronts, which feed the MFMAs from memory without a barrier; the
// NW partial tiles are added through LDS in wavefront order, so the sum order is fixed by the shape. The large-tile kernels need a
// grid of 64 x 64 tiles to fill the chip, split tiles and add them up in a second launch where it does not, and take operands
// whose K is ragged through registers element by element or from a transposed copy; here any K and both forms of each operand cost the
// same.
//
// An operand whose K is contiguous is loaded 64 bytes of a row at a time by four neighbouring lanes (in the MFMA layout
// neighbouring lanes read different rows, and a compute unit then takes in 16 bytes a cycle instead of 64) and turned into the
// MFMA layout through the wavefront's own LDS, whose instructions execute in order; one whose rows or columns are contiguous is in
// that layout as it is read. A group is 8 k: lane group g of the wavefront holds k 2 g and 2 g + 1 of it. U groups are in flight.
// SHORT: chains of 16 MFMAs are added to a sum with ordinary additions, so that the error does not grow with the root of K: a chain
// of L MFMAs loses 9.6e-17 sqrt(L / 2). It is for few tiles, whose K the large-tile kernels cut over many workgroups. Relative
// 2-norm error against extended precision, those kernels / one chain a wavefront / here: 64 x 600 x 1500 3.3e-16 / 4.8e-16 / 2.9e-16, 300 x 900 x
// 2500 6.3e-16 / 8.2e-16 / 3.0e-16; us without and with it 17.7 / 17.7 (A stored [k, m] 18.4 / 19.4), 300 x 300 x 1500 21.0 / 22.4, 512^3 10.5 / 10.8.
// Bound by the matrix units and the vector instructions that share their issue cycles: 1500^3 41 of the 78.6 TFLOP/s.

#include "devmath.hpp"
#include "gemm_f64.hpp"

namespace {

using D2 = __attribute__((ext_vector_type(2))) double;
typedef D2 D2_any __attribute__((aligned(8)));  // 128-bit access at any double
using D4 = __attribute__((ext_vector_type(4))) double;

constexpr int kXcds = 8;

// KA, KB: K is the contiguous direction of A, of B.
// Three wavefronts a SIMD are asked for where that keeps the accumulators out of the second half of the register file: without it 64
// moves between the halves surround every 16 MFMAs and share their issue cycles (1000 x 1024 x 1021 with A stored [k, m] 53.9 -> 53.0 us,
// 620 x 1572 x 1768 83.6 -> 75.9; 1021 x 1024 x 1000 53.5 -> 48.5). With B stored [n, k] its loads then lie closer to their use and rows
// of odd length lose more than the moves cost (1524 x 1997 x 1375 221 -> 250), so that form stays as the compiler lays it out.
template <int NW, int U, bool SHORT, bool KA, bool KB>
__global__ __launch_bounds__(64 * NW, NW == 4 && !KB ? 3 : 1) void gemm_f64_kernel(const fth::SmallGemm64 p, const int tiles_m, const int tiles_n) {
    constexpr int T = 2, TILE = 1024, STAGED = T * ((KA ? 1 : 0) + (KB ? 1 : 0)), SLOT = STAGED * TILE;  // a tile: 16 rows x 64 bytes
    constexpr int PART = T * T * 4 * 64 * 8;  // a wavefront's partial tile, in its accumulator layout
    constexpr int AREA = 2 * SLOT > PART ? 2 * SLOT : PART;
    __shared__ __attribute__((aligned(16))) unsigned char smem[NW][AREA];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, g = lane >> 4, qrow = lane >> 2, qc = lane & 3;
    // The row tiles of one column tile are eight workgroups apart, on one XCD.
    const int run = kXcds * tiles_m, first_n = (int)blockIdx.x / run * kXcds, in_run = (int)blockIdx.x % run;
    const int width = tiles_n - first_n < kXcds ? tiles_n - first_n : kXcds;
    const int tile_m = in_run / width, tile_n = first_n + in_run % width;
    const int64_t batch = blockIdx.y, m0 = (int64_t)tile_m * 32, n0 = (int64_t)tile_n * 32;
    // whole groups, contiguous for each wavefront, in wavefront order; what is left of K goes to the last wavefront
    const int groups = (int)(p.k / 8), rest = (int)(p.k % 8), per = (groups + NW - 1) / NW;
    const int g0 = wave * per, g1 = g0 + per < groups ? g0 + per : groups, last = groups > 0 ? groups - 1 : 0;
    const double *ap[T], *bp[T];  // this lane's first two k; rows and columns past the edge repeat the last one and are never stored
#pragma unroll
    for (int i = 0; i < T; ++i) {
        int64_t row = m0 + i * 16 + (KA ? qrow : l16), col = n0 + i * 16 + (KB ? qrow : l16);
        row = row < p.m ? row : p.m - 1;
        col = col < p.n ? col : p.n - 1;
        ap[i] = p.a + batch * p.stride_a + (KA ? row * p.lda : row);
        bp[i] = p.b + batch * p.stride_b + (KB ? col * p.ldb : col);
    }
    const int64_t a_lane = KA ? 2 * qc : 2 * g * p.lda, b_lane = KB ? 2 * qc : 2 * g * p.ldb;
    const int64_t a_step = KA ? 8 : 8 * p.lda, b_step = KB ? 8 : 8 * p.ldb;
    D2 av[U][T], bv[U][T];
    auto load = [&](int u, int group) __attribute__((always_inline)) {
        const int64_t t = group < last ? group : last;
#pragma unroll
        for (int i = 0; i < T; ++i) {
            const double *a = ap[i] + a_lane + t * a_step, *b = bp[i] + b_lane + t * b_step;
            if (KA) av[u][i] = *reinterpret_cast<const D2_any *>(a);
            else av[u][i] = D2{a[0], a[p.lda]};
            if (KB) bv[u][i] = *reinterpret_cast<const D2_any *>(b);
            else bv[u][i] = D2{b[0], b[p.ldb]};
        }
    };
    // The last K % 8: two k of a row, or of a column, each on its own and zero past the end.
    auto load_rest = [&](D2 (&v)[T], const double *const (&src)[T], bool by_k, int64_t ks) __attribute__((always_inline)) {
        const int64_t k = (int64_t)groups * 8 + 2 * (by_k ? qc : g);
#pragma unroll
        for (int i = 0; i < T; ++i) v[i] = D2{k < p.k ? src[i][k * ks] : 0.0, k + 1 < p.k ? src[i][(k + 1) * ks] : 0.0};
    };
    unsigned char *area = smem[wave];
    const int wr = qrow * 64 + ((qc ^ fth::swz(qrow)) << 4), rd = l16 * 64 + ((g ^ fth::swz(l16)) << 4);
    auto stage = [&](int u) __attribute__((always_inline)) {
        unsigned char *s = area + (u & 1) * SLOT + wr;
#pragma unroll
        for (int i = 0; i < T; ++i) {
            if (KA) *reinterpret_cast<D2 *>(s + i * TILE) = av[u][i];
            if (KB) *reinterpret_cast<D2 *>(s + ((KA ? T : 0) + i) * TILE) = bv[u][i];
        }
    };
    D4 acc[T][T], sum[T][T];
    auto clear = [](D4 (&x)[T][T]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < T; ++i)
#pragma unroll
            for (int j = 0; j < T; ++j) x[i][j] = D4{0.0, 0.0, 0.0, 0.0};
    };
    auto collect = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < T; ++i)
#pragma unroll
            for (int j = 0; j < T; ++j) sum[i][j] += acc[i][j];
    };
    clear(acc);
    if (SHORT) clear(sum);
    auto multiply = [&](int u, D2 (&a)[T], D2 (&b)[T]) __attribute__((always_inline)) {
        const unsigned char *s = area + (u & 1) * SLOT + rd;
#pragma unroll
        for (int i = 0; i < T; ++i) {
            if (KA) a[i] = *reinterpret_cast<const D2 *>(s + i * TILE);
            if (KB) b[i] = *reinterpret_cast<const D2 *>(s + ((KA ? T : 0) + i) * TILE);
        }
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int i = 0; i < T; ++i)
#pragma unroll
                for (int j = 0; j < T; ++j) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i][e], b[j][e], acc[i][j], 0, 0, 0);
    };
    if (g0 < g1) {
#pragma unroll
        for (int u = 0; u < U; ++u) load(u, g0 + u);
    }
    int t0 = g0;
    for (; t0 + U < g1; t0 += U) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            stage(u);
            D2 a[T], b[T];
#pragma unroll
            for (int i = 0; i < T; ++i) {
                a[i] = av[u][i];
                b[i] = bv[u][i];
            }
            load(u, t0 + U + u);
            multiply(u, a, b);
        }
        if (SHORT && ((t0 - g0) & (8 - U)) == 8 - U) {  // every eight groups
            collect();
            clear(acc);
        }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (t0 + u < g1) {
            stage(u);
            multiply(u, av[u], bv[u]);
        }
    if (rest != 0 && wave == NW - 1) {
        load_rest(av[0], ap, KA, KA ? 1 : p.lda);
        load_rest(bv[0], bp, KB, KB ? 1 : p.ldb);
        stage(0);
        multiply(0, av[0], bv[0]);
    }
    if (SHORT) collect();
    double *part = reinterpret_cast<double *>(area);
#pragma unroll
    for (int i = 0; i < T; ++i)
#pragma unroll
        for (int j = 0; j < T; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) part[((i * T + j) * 4 + r) * 64 + lane] = SHORT ? sum[i][j][r] : acc[i][j][r];
    __syncthreads();
    double *C = p.c + batch * p.stride_c;
    for (int e = wave; e < T * T * 4; e += NW) {  // accumulator element r of a lane: row 4 r + lane / 16, column lane % 16
        const int64_t row = m0 + (e / (4 * T)) * 16 + 4 * (e & 3) + g, col = n0 + (e / 4 % T) * 16 + l16;
        if (row >= p.m || col >= p.n) continue;
        double v = reinterpret_cast<const double *>(smem[0])[e * 64 + lane];
#pragma unroll
        for (int w = 1; w < NW; ++w) v += reinterpret_cast<const double *>(smem[w])[e * 64 + lane];
        if (p.alpha != 1.0) v = p.alpha * v;
        if (p.epilogue & FTH_EPI_BIAS) v = v + p.bias[col];
        if (p.epilogue & FTH_EPI_GELU) v = fth::gelu_erf(v);
        if (p.epilogue & FTH_EPI_GELU_TANH) v = fth::gelu_tanh(v);
        if (p.epilogue & FTH_EPI_RESIDUAL) v = v + p.residual[batch * p.stride_c + row * p.ldc + col];
        C[row * p.ldc + col] = v;
    }
}

template <int NW, int U, bool SHORT, bool KA, bool KB> int32_t launch(const fth::SmallGemm64 &g, hipStream_t st) {
    const int tiles_m = (int)fth::ceil_div(g.m, 32), tiles_n = (int)fth::ceil_div(g.n, 32);
    // Four workgroups fit on a compute unit in this form; with a long K and more than one round of them, three share L2 better
    // (us with four / three: 1500^3 181 / 167, 4001 x 4001 x 999 797 / 748; in one round 1021 x 1024 x 1000 48.8 / 52.1; with a short K
    // 8000 x 500 x 250 60.9 / 65.4, 1768 x 1572 x 620 85 / 86), for which each takes 48 of the 160 KB of LDS.
    const unsigned reserve = NW == 4 && KA && !KB && g.k >= 800 && (int64_t)tiles_m * tiles_n * g.batch > 1024 ? 16384 : 0;
    gemm_f64_kernel<NW, U, SHORT, KA, KB><<<dim3((unsigned)(tiles_m * tiles_n), (unsigned)g.batch), dim3(64 * NW), reserve, st>>>(g, tiles_m, tiles_n);
    FTH_CHECK_LAUNCH("gemm_f64");
    return FTH_OK;
}

template <bool KA, bool KB> int32_t choose(const fth::SmallGemm64 &g, hipStream_t st) {
    // Few tiles: eight wavefronts share K, four groups ahead (512^3 8.9 us, four wavefronts 10.5); otherwise four, with fewer registers
    // and so more workgroups on a compute unit (1500^3 166 us, eight wavefronts 190).
    const int64_t tiles = fth::ceil_div(g.m, 32) * fth::ceil_div(g.n, 32) * g.batch;
    if (tiles <= 256) return launch<8, 4, true, KA, KB>(g, st);
    // The large-tile kernels cut K of about as many tiles; from 512 on they walk it in one chain, with more error than four (1021 x 1024 x
    // 1000 7.3e-16 / 5.4e-16), and the registers of the sum would cost a workgroup of the four on a compute unit.
    return tiles <= 512 ? launch<4, 2, true, KA, KB>(g, st) : launch<4, 2, false, KA, KB>(g, st);
}

}  // namespace

namespace fth {

bool small_gemm_f64(const SmallGemm64 &g, hipStream_t st, int32_t *rc) {
    const int64_t tiles = ceil_div(g.m, 32) * ceil_div(g.n, 32) * g.batch, tiles64 = ceil_div(g.m, 64) * ceil_div(g.n, 64) * g.batch;
    if (g.k < 2 || g.batch > 65535 || ceil_div(g.m, 32) * ceil_div(g.n, 32) > (1 << 24)) return false;
    // Where it is the fastest, us of the large-tile kernels / here. K has to be short enough for its share of a few wavefronts (512 x 512
    // x 2048 30.5 / 24.2, but 300 x 300 x 5001 45 / 63). Operands that go straight to LDS there (K in whole K-tiles, aligned rows): until
    // 64 x 64 tiles fill the chip (512^3 20.5 / 9.7, 768 x 1024 x 1024 39.3 / 35.5, but 896^3 37.9 / 41.1, 1024^3 45 / 48, 2048^3 261 / 332),
    // later with a short K (1024 x 1024 x 128 20.9 / 12.4; 2048 x 1024 x 128 16.4 / 19.1). All others at any size: 1000 x 1024 x 1021 with A stored
    // [k, m] 73.8 / 52.7, 1021 x 1024 x 1000 65 / 52, 3001 x 3000 x 301 180 / 153, 4001 x 4001 x 999 834 / 819, 300 x 300 x 9 26 / 4.3.
    // Two corners are slower: a very few tiles with a long K that goes straight to LDS there (64 x 64 x 2000 20.5 / 21.3 to 23.9 by form, 64 x
    // 64 x 1408 16.9 / 16.0 to 18.2, 17 x 290 x 2000 22.5 / 21.4), and with both K contiguous a long K on few tiles more than one for
    // every compute unit (300 x 900 x 2500 50.2 / 60.1, 1700 38.8 / 41.3, 1300 33.0 / 32.3; 450 x 1000 x 2500 72 / 64).
    if (g.k > (tiles <= 256 ? 2048 : 2560) || (g.trans_b && g.k > 1600 && tiles > 256 && tiles <= 320)) return false;
    auto even = [](int64_t ld, int64_t stride, const double *x) { return ld % 2 == 0 && stride % 2 == 0 && (reinterpret_cast<uintptr_t>(x) & 15u) == 0; };
    const bool direct = g.k % 16 == 0 && even(g.lda, g.stride_a, g.a) && even(g.ldb, g.stride_b, g.b) && (!g.trans_a || g.m % 2 == 0) && (g.trans_b || g.n % 2 == 0);
    if (direct && tiles <= 8 && g.k > 1536) return false;
    if (direct && g.k > 64 && tiles > 256 && !(g.k <= 1024 && tiles64 <= 192) && !(g.k <= 256 && tiles64 <= 256)) return false;
    const bool ka = !g.trans_a, kb = g.trans_b;
    if (!ka && kb) return false;  // (the entry point refuses this form)
    *rc = !ka ? choose<false, false>(g, st) : kb ? choose<true, true>(g, st) : choose<true, false>(g, st);
    return true;
}

}  // namespace fth
