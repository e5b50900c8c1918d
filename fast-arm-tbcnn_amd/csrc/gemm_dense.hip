// fp32 GEMM, C = alpha * op(A) * op(B) + beta * Cin, on v_mfma_f32_16x16x4_f32
// (tbn::gemm, gemm.cpp:349-360).
//
// Order of the sum.  Chain c (0..3) of an output runs over the 4-value groups
// c, c + 4, c + 8, ... of k, one fp32 FMA after the other in ascending k, and
// the result is (chain 0 + chain 1) + (chain 2 + chain 3).  On gfx950 the
// matrix instruction gives exactly those bits: its four products are added to
// the accumulator one at a time, ascending, each with one rounding
// (compared bit by bit with fmaf over 2e7 results, subnormals, infinities and
// NaN included), so one instruction is one group of one chain.
//
// A block owns a T x T tile of C; its four waves own one chain each of the
// whole tile, so a small product still gives every SIMD work, and a wave
// reads an operand value from LDS once for T / 16 instructions.  Chunks of
// the tile's rows of op(A) and columns of op(B) are staged as fp32 in two LDS
// buffers; an operand keeps the order it has in memory, rows of contiguous k
// or (transposed) rows of contiguous columns, and both pitches keep the 64
// lanes' reads on different banks.
//
// What bounds it: the fp32 matrix pipe (157 TFLOP/s dense) for large products,
// latency for small ones.  Measured (kernel time): 2048^3 150-164 us = 105-114
// TFLOP/s; 1024 x 1024 x 1000 24.9 us with op(B) stored [N, K] and 29.1 with
// [K, N] (126 and 176 us as one 16 x 4 tile of fp32 FMA chains per block, the
// kernel this replaces, whose bits it keeps); the ResNet-18 classifier (32 x
// 512 x 1000) 4.2 us (5.2).  The six bf16 products that stand for one fp32
// product have a 2.6 times higher peak, but round each product and cost three
// times the LDS traffic and a split of both operands.
#include <type_traits>

#include "dense_core.hpp"
#include "gemm_dense.hpp"

namespace {

using namespace tbnk;

template <class Tile, bool A_KCONT, bool B_KCONT>
__global__ void __launch_bounds__(256, 2) gemm_dense_kernel(tbn_hip::DenseGemmArgs g, int tiles_r, int tiles_c) {
    constexpr int T = Tile::T, F = T / 16;
    constexpr int kA = Tile::operand(A_KCONT), kBuffer = kA + Tile::operand(B_KCONT);
    constexpr int kSums = 4 * T * Tile::RPITCH;
    __shared__ __attribute__((aligned(16))) float lds[2 * kBuffer > kSums ? 2 * kBuffer : kSums];
    int tr, tc;
    tile_coords(tiles_r, tiles_c, tr, tc);
    const int m0 = tr * T, n0 = tc * T;
    const int tid = static_cast<int>(threadIdx.x);
    const int lane = tid & 63, chain = tid >> 6;

    f32x4_t acc[F][F];
#pragma unroll
    for (int i = 0; i < F; ++i)
#pragma unroll
        for (int j = 0; j < F; ++j) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

    const DenseOperand<Tile, A_KCONT> oa(g.A, A_KCONT ? g.a_row : g.a_k, m0, g.M, g.K);
    const DenseOperand<Tile, B_KCONT> ob(g.B, B_KCONT ? g.b_col : g.b_k, n0, g.N, g.K);
    // chunk ch sits in LDS buffer ch & 1; chunk ch + 1 is fetched into registers
    // as chunk ch's instructions start and stored after them (two chunks ahead
    // measured the same and costs registers)
    f32x4_t av[Tile::PER], bv[Tile::PER];
    oa.load(av, 0);
    ob.load(bv, 0);
    oa.store(lds, av, 0, g.K);
    ob.store(lds + kA, bv, 0, g.K);
    __syncthreads();
    const int chunks = (g.K + Tile::KC - 1) / Tile::KC;
    for (int ch = 0; ch < chunks; ++ch) {
        const float* buf = lds + (ch & 1) * kBuffer;
        const int k1 = (ch + 1) * Tile::KC;
        if (k1 < g.K) {
            oa.load(av, k1);
            ob.load(bv, k1);
        }
        dense_multiply<Tile, A_KCONT, B_KCONT>(buf, chain, lane, acc);
        if (k1 < g.K) {
            float* next = lds + ((ch + 1) & 1) * kBuffer;
            oa.store(next, av, k1, g.K);
            ob.store(next + kA, bv, k1, g.K);
        }
        __syncthreads();
    }

    // the four chains through LDS; a thread then finishes 4 consecutive
    // columns of a row
    dense_put_chain<Tile>(lds, chain, lane, acc);
    __syncthreads();
#pragma unroll
    for (int i = tid; i < T * T / 4; i += 256) {
        const int r = i / (T / 4), c = (i % (T / 4)) * 4;
        const int m = m0 + r, n = n0 + c;
        if (m >= g.M || n >= g.N) continue;
        f32x4_t y = dense_sum_chains<Tile>(lds, r, c);
        float* out = g.out + static_cast<int64_t>(m) * g.N + n;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float v = y[e] * g.alpha + 0.0f;
            if (g.cin) {
                const int nc = min(n + e, g.N - 1);
                v += g.beta * (g.cin_1d ? g.cin[nc] : g.cin[static_cast<int64_t>(m) * g.N + nc]);
            }
            if (g.flags & TBN_EPI_RELU) v = v > 0.0f ? v : 0.0f;
            y[e] = v;
        }
        if (n + 4 <= g.N) {
            *reinterpret_cast<f32x4u_t*>(out) = y;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (n + e < g.N) out[e] = y[e];
        }
    }
}

template <class Tile>
int launch_dense(const tbn_hip::DenseGemmArgs& a, hipStream_t s) {
    const int64_t tiles_r = tbn_hip::ceil_div(a.M, Tile::T), tiles_c = tbn_hip::ceil_div(a.N, Tile::T);
    TBN_REQUIRE(tiles_r * tiles_c < (1LL << 31), TBN_INVALID_SHAPE, "too many tiles");
    const dim3 grid(static_cast<unsigned>(tiles_r * tiles_c));
    auto launch = [&](auto ak, auto bk) {
        hipLaunchKernelGGL((gemm_dense_kernel<Tile, decltype(ak)::value, decltype(bk)::value>), grid, dim3(256), 0, s,
                           a, static_cast<int>(tiles_r), static_cast<int>(tiles_c));
    };
    using KCont = std::true_type;
    using CCont = std::false_type;
    if (a.a_k == 1) a.b_k == 1 ? launch(KCont{}, KCont{}) : launch(KCont{}, CCont{});
    else a.b_k == 1 ? launch(CCont{}, KCont{}) : launch(CCont{}, CCont{});
    return tbn_hip::check_launch("gemm_f32 (dense)");
}

}  // namespace

namespace tbn_hip {

// The tile only decides how the work is spread; every tile gives the same
// bits, so M may take part.  Two blocks of the 64 x 64 tile fit a CU; it moves
// the fewest operand bytes per product and is the fastest when its last round
// of 512 blocks is nearly full (1024 x 2048, K 1024: 41.8 us against 46.1 for
// 32 x 32), not otherwise (1500 x 2000, K 700: 58.9 against 50.9).  From 256
// tiles of 32 x 32 (one per CU) on, that tile (512 x 512, K 1024: 9.6 us against 12.4 for
// 16 x 16); below, 16 x 16 (322 x 301, K 1146: 8.6 against 12.9), with long
// chunks, for fewer barriers, while two blocks per CU hold all of them (256 x
// 512, K 1024: 7.2 us against 7.6), else shorter ones, so that four blocks fit a
// CU (700 x 600, K 300: 9.8 against 14.9).
int gemm_dense(const DenseGemmArgs& a, hipStream_t stream) {
    auto tiles = [&](int64_t t) { return ceil_div(a.M, t) * ceil_div(a.N, t); };
    const int64_t big = tiles(64);
    if (big >= 0.9 * 512 * ceil_div(big, 512)) return launch_dense<DenseTile<64, 64>>(a, stream);
    if (tiles(32) >= 256) return launch_dense<DenseTile<32, 64>>(a, stream);
    if (tiles(16) > 512) return launch_dense<DenseTile<16, 128>>(a, stream);
    return launch_dense<DenseTile<16, 256>>(a, stream);
}

}  // namespace tbn_hip
