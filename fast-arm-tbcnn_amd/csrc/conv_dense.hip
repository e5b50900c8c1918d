// fp32 Conv2D (tbn::conv2d, conv2d.cpp:78-192) as an implicit GEMM on the fp32
// matrix instructions.
//
// The product W[M, K] * X[K, Q], k = (c, r, s) and Q the output positions, runs
// like gemm_dense.hip's: T x T tiles of (channels, positions), chunks of k
// staged as fp32 in two LDS buffers, one chain of 4-value groups of k per
// wave, so every tile gives the same bits and a sample's result does not
// depend on its batch.  X is gathered while it is staged: a thread owns one
// position, whose input offset and whose taps inside the image (a bit each) it
// works out once, and loads one value per k; taps outside the image, and
// k >= K, get an offset past the buffer's range and read as zero.  With the fused
// 2x2 pool the positions run window by window, so the four consecutive positions
// that a thread finishes are one window.
//
// What bounds it: the fp32 matrix pipe (157 TFLOP/s dense) for large layers, the
// gather's vector instructions beside it.  Measured (us a pass; before
// = a 64 x 64 tile of six bf16 products per fp32 one, gathered and split in every
// 32-k step, or one output per thread for the smallest): 16 x 128 x 28 x 28 ->
// 128, 3x3, 57.7 (83.5 before), 32 x 64 x 56 x 56 -> 64 101 (113), 4 x 31 x 17 x 17
// -> 24, 5x5, 9.3 (75.8), 1 x 512 x 7 x 7 -> 512 29.7 (282), 64 x 100 x 7 x 7 -> 100 22 (72),
// 1 x 6 x 12 x 12 -> 16, 5x5, 5.3 (6.4); the error against 64 bits is about half.
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "conv_common.hpp"
#include "dense_core.hpp"

namespace {

using namespace tbnk;

struct DenseConv {
    const float* x;
    const float* w;     // [M, K]
    const float* bias;  // may be null
    float* y;
    ConvGeom g;
    int N, M, taps;
    int flags;
    UDiv div_taps, div_kw;
};

template <class Tile>
__global__ void __launch_bounds__(256, 2) conv_dense_kernel(DenseConv p, int tiles_r, int tiles_c) {
    constexpr int T = Tile::T, KC = Tile::KC;
    constexpr int kA = Tile::operand(true), kBuffer = kA + Tile::operand(false);
    constexpr int kSums = 4 * T * Tile::RPITCH;
    constexpr int PER = T * KC / 256;   // values of X a thread stages per chunk
    constexpr int KROWS = 256 / T;      // rows of k the block loads at once
    __shared__ __attribute__((aligned(16))) float lds[2 * kBuffer > kSums ? 2 * kBuffer : kSums];
    const ConvGeom& g = p.g;
    int tr, tc;
    tile_coords(tiles_r, tiles_c, tr, tc);
    const int m0 = tr * T, q0 = tc * T;
    const int tid = static_cast<int>(threadIdx.x);
    const int lane = tid & 63;
    const int chain = __builtin_amdgcn_readfirstlane(tid >> 6);

    f32x4_t acc[T / 16][T / 16];
#pragma unroll
    for (int i = 0; i < T / 16; ++i)
#pragma unroll
        for (int j = 0; j < T / 16; ++j) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

    // this thread's position: offset of its window's first tap from the
    // tile's first image, and a bit per tap inside the image
    int n, oh, ow, n0;
    position_coords(g, q0, n0, oh, ow);
    position_coords(g, min(q0 + tid % T, g.Q - 1), n, oh, ow);
    const int ih0 = oh * g.sh - g.ph, iw0 = ow * g.sw - g.pw;
    const int hw = g.H * g.W;
    const int at = ((n - n0) * g.C * hw + ih0 * g.W + iw0) * 4;
    uint32_t outside = 0x80000000u;  // bit 31: k >= K
    for (int r = 0; r < g.kh; ++r)
        for (int s = 0; s < g.kw; ++s) {
            const int ih = ih0 + r * g.dh, iw = iw0 + s * g.dw;
            const bool in = static_cast<unsigned>(ih) < static_cast<unsigned>(g.H) &&
                            static_cast<unsigned>(iw) < static_cast<unsigned>(g.W);
            outside |= (in ? 0u : 1u) << (r * g.kw + s);
        }
    const int64_t image = static_cast<int64_t>(g.C) * hw;
    const uint64_t left = static_cast<uint64_t>(p.N - n0) * image * 4;
    // offsets stay below 2^31 (host-checked), so the one that means "outside" is past any range
    const __amdgpu_buffer_rsrc_t rs = buffer_range(p.x + n0 * image, left < 0x7FFFFFFFull ? left : 0x7FFFFFFFull, 0);

    const DenseOperand<Tile, true> ow_(p.w, g.K, m0, p.M, g.K);
    f32x4_t wv[Tile::PER];
    float xv[PER];
    // (byte offset of (c, r, s) from a window's first tap, tap) of a chunk's k,
    // worked out by one thread per k two chunks ahead
    __shared__ int2 table[2][KC];
    auto put_table = [&](int ch) {
        if (tid < KC) {
            const int k = ch * KC + tid;
            const int c = udiv(k, p.div_taps);
            const int tap = k - c * p.taps;
            const int r = udiv(tap, p.div_kw);
            const int off = c * hw + r * g.dh * g.W + (tap - r * g.kw) * g.dw;
            table[ch & 1][tid] = k < g.K ? make_int2(off * 4, tap) : make_int2(0, 31);
        }
    };
    const int krow = tid / T;
    auto load_x = [&](int ch) {
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int2 e = table[ch & 1][j * KROWS + krow];
            // the tap's bit spread over the word: an offset past any range outside the image
            const uint32_t out = static_cast<uint32_t>(static_cast<int>(outside << (31 - e.y)) >> 31);
            const uint32_t voff = (out & 0x80000000u) | static_cast<uint32_t>(at + e.x);
            xv[j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, voff, 0, 0));
        }
    };
    auto store_x = [&](float* buf) {
#pragma unroll
        for (int j = 0; j < PER; ++j) buf[kA + (j * KROWS + krow) * Tile::CPITCH + tid % T] = xv[j];
    };

    put_table(0);
    put_table(1);
    __syncthreads();
    ow_.load(wv, 0);
    load_x(0);
    ow_.store(lds, wv, 0, g.K);
    store_x(lds);
    __syncthreads();
    const int chunks = (g.K + KC - 1) / KC;
    for (int ch = 0; ch < chunks; ++ch) {
        const int k1 = (ch + 1) * KC;
        if (k1 < g.K) {
            ow_.load(wv, k1);
            load_x(ch + 1);
            put_table(ch + 2);
        }
        dense_multiply<Tile, true, false>(lds + (ch & 1) * kBuffer, chain, lane, acc);
        if (k1 < g.K) {
            float* next = lds + ((ch + 1) & 1) * kBuffer;
            ow_.store(next, wv, k1, g.K);
            store_x(next);
        }
        __syncthreads();
    }

    dense_put_chain<Tile>(lds, chain, lane, acc);
    __syncthreads();
    const bool relu = (p.flags & TBN_EPI_RELU) != 0;
#pragma unroll
    for (int i = tid; i < T * T / 4; i += 256) {
        const int row = i / (T / 4), c = (i % (T / 4)) * 4;
        const int m = m0 + row, q = q0 + c;
        if (m >= p.M || q >= g.Q) continue;
        const float b = p.bias ? p.bias[m] : 0.0f;
        f32x4_t v = dense_sum_chains<Tile>(lds, row, c);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] += b;
            if (relu) v[e] = v[e] > 0.0f ? v[e] : 0.0f;
        }
        if (g.pool) {
            // Q is a multiple of 4 and q of a window
            const int win = q >> 2, img = win / g.PHW;
            p.y[(static_cast<int64_t>(img) * p.M + m) * g.PHW + (win - img * g.PHW)] =
                fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3]));
            continue;
        }
        const int img = q / g.OHW, at_y = q - img * g.OHW;
        float* out = p.y + (static_cast<int64_t>(img) * p.M + m) * g.OHW + at_y;
        if (at_y + 4 <= g.OHW) {
            *reinterpret_cast<f32x4u_t*>(out) = v;
        } else {
            // the four positions reach into the next image(s) or past the last
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (q + e >= g.Q) break;
                const int im = (q + e) / g.OHW;
                p.y[(static_cast<int64_t>(im) * p.M + m) * g.OHW + (q + e - im * g.OHW)] = v[e];
            }
        }
    }
}

template <class Tile>
int launch_conv_dense(const DenseConv& p, hipStream_t s) {
    const int64_t tiles_r = tbn_hip::ceil_div(p.M, Tile::T), tiles_c = tbn_hip::ceil_div(p.g.Q, Tile::T);
    TBN_REQUIRE(tiles_r * tiles_c < (1LL << 31), TBN_INVALID_SHAPE, "too many tiles");
    hipLaunchKernelGGL(conv_dense_kernel<Tile>, dim3(static_cast<unsigned>(tiles_r * tiles_c)), dim3(256), 0, s, p,
                       static_cast<int>(tiles_r), static_cast<int>(tiles_c));
    return tbn_hip::check_launch("conv2d_f32 (dense)");
}

}  // namespace

namespace tbn_hip {

// One image's shape decides (not the batch): enough k for a chunk of 64 or
// more (at K = 4 a 7 x 4 x 96 x 96 -> 324 layer takes 73.7 us here and 52.2 with the
// gathered bf16 splits of conv.hip), a bit per tap, and lane offsets
// of the images a tile can touch below 2^31 bytes.
bool conv_dense_supported(const tbn_conv2d_desc* d) {
    const int64_t oh = (d->h + 2 * d->ph - d->dh * (d->kh - 1) - 1) / d->sh + 1;
    const int64_t ow = (d->w + 2 * d->pw - d->dw * (d->kw - 1) - 1) / d->sw + 1;
    const int64_t plane = std::max<int64_t>(1, (oh / 2) * (ow / 2) * 4);  // positions of an image, pooled or not, at least
    const int64_t images = 64 / plane + 2;
    // rows and columns of the padding count as offsets too
    const int64_t reach = (d->c * d->h + d->ph + d->dh * d->kh) * (d->w + d->pw + d->dw * d->kw);
    return d->c * d->kh * d->kw > 32 && d->kh * d->kw <= 31 && d->m < (1LL << 31) && images * reach * 4 < (1LL << 31) &&
           64 * d->c * d->kh * d->kw * 4 < (1LL << 31);
}

int conv_dense_run(const float* x, const tbn_conv2d_desc* d, const float* w, const float* bias, int flags, float* y,
                   hipStream_t stream) {
    DenseConv p{x, w, bias, y, {}, static_cast<int>(d->n), static_cast<int>(d->m),
                static_cast<int>(d->kh * d->kw), flags, make_udiv(static_cast<uint32_t>(d->kh * d->kw)),
                make_udiv(static_cast<uint32_t>(d->kw))};
    if (int rc = make_geom(d, flags, p.g)) return rc;
    auto tiles = [&](int64_t t) { return ceil_div(p.M, t) * ceil_div(p.g.Q, t); };
    // The tile only decides how the work is spread.  64 x 64 moves the fewest
    // values per product (16 x 128 x 28 x 28 -> 128, 3x3, 57.7 us against 67.8
    // for 32 x 32) while it gives most CUs a block and its rows are not half
    // empty; 32 x 32 next (16 x 32 x 28 x 28 -> 32, 5x5, 19.0 us against 22.5
    // for 16 x 16); 16 x 16 for what is left (2 x 128 x 28 x 28 -> 128 15.7 us
    // against 18.4, 1 x 512 x 7 x 7 -> 512 29.7 against 63.9).
    if (p.M > 32 && tiles(64) >= 190) return launch_conv_dense<DenseTile<64, 64>>(p, stream);
    if (p.M > 16 && tiles(32) >= 256) return launch_conv_dense<DenseTile<32, 64>>(p, stream);
    return launch_conv_dense<DenseTile<16, 128>>(p, stream);
}

}  // namespace tbn_hip
