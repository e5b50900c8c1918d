// float x binary / ternary GEMM with K split over the waves of a block, for
// products whose tiles are too few, or whose K is too long, for the staged
// tiles of gemm_wide.hip (a layer at a small or serving batch).
//
// A block owns one small tile of C: 16 or 32 rows of A (one matrix
// instruction) x 1 to 4 fragments of as many columns.  Each of its 4 or 8
// waves runs a contiguous part of K on the whole tile by itself, without a
// barrier: it loads its 32 k of the rows (16 bytes a lane, whole 128-byte lines),
// turns them round through its own LDS rows so that a lane holds its row's
// values, splits them into three bf16 parts (hi + mid + lo = a exactly) and
// multiplies them by the weights, decoded from the packed words in
// registers; the loads run three steps ahead.  The waves' sums are
// added in wave order through LDS.  So a product of one row and 4096 columns
// gives 256 CUs eight waves each, and nothing passes through memory between
// blocks: no workspace, and the call may be captured.
//
// What bounds it: vector instructions.  A SIMD's 32x32x16 instruction leaves
// room for about 6 of them; a step's split costs 120 and a fragment's decode
// 17 (two shifts-and-masks per dword of two weights: the order of k inside a
// step is chosen so that a dword's two weights are 16 bits apart).  More
// columns per tile share the split, fewer give more blocks.
//
// Measured (kernel time, us; before = one 64 x 64 tile per block over the
// whole of K, or K split over blocks through memory): 1 x 4096 x 4096 9.0
// (81.7 before), 24 x 4096 x 4096 10.6 (94.2), 64 x 4096 x 4096 13.4 (23.3),
// 291 x 410 x 383 5.1 (16.8), 128 x 1024 x 4096 8.6 (18.2), 777 x 1333 x 1001 14.3 (28.2),
// 256 x 4096 x 4096 29.5, ternary 32.1 (34.0, 36.7), 2000^3 54.9 (60.0).
#include <algorithm>
#include <string>
#include <type_traits>

#include "gemm_wide.hpp"
#include "mfma_core.hpp"

namespace {

using namespace tbnk;

typedef float f32x4_t __attribute__((ext_vector_type(4)));

template <int ROWS_, int CT_, int KG_>
struct WavesCfg {
    static constexpr int ROWS = ROWS_;       // rows of the tile: 32 (32x32x16 instructions) or 16 (16x16x32)
    static constexpr int CT = CT_;           // column fragments of ROWS columns
    static constexpr int KG = KG_;           // waves, each with a contiguous part of K
    static constexpr int NT = 64 * KG;
    static constexpr int BC = ROWS * CT;
    static constexpr int SL = ROWS / 16;     // k slices (instructions per plane and fragment) per step of 32 k
    static constexpr int ACC = ROWS * ROWS / 64;
    static constexpr int P = CT >= 2 && KG * ROWS * ROWS <= 8192 ? 2 : 1;  // fragments summed per pass
    static constexpr int STAGE = ROWS * 32;  // floats a wave stages per step
    static constexpr int LDS = KG * (P * ROWS * ROWS > STAGE ? P * ROWS * ROWS : STAGE);
    static_assert(ROWS == 32 || ROWS == 16, "one matrix instruction covers the tile's rows");
};

template <class Cfg>
struct WavesAcc;
template <int CT, int KG>
struct WavesAcc<WavesCfg<32, CT, KG>> {
    using type = f32x16_t;
    static __device__ __forceinline__ type mfma(u32x4_t a, u32x4_t b, type c) { return mfma32(a, b, c); }
    static __device__ __forceinline__ int row(int e, int lane) { return 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3); }
};
template <int CT, int KG>
struct WavesAcc<WavesCfg<16, CT, KG>> {
    using type = f32x4_t;
    static __device__ __forceinline__ type mfma(u32x4_t a, u32x4_t b, type c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                       __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int e, int lane) { return 4 * (lane >> 4) + e; }
};

template <class Cfg, bool TERNARY>
__global__ void __launch_bounds__(Cfg::NT)
gemm_waves_kernel(tbn_hip::WideGemmArgs p, int tiles_r, int tiles_c, int per_xcd, int group_r) {
    __shared__ __attribute__((aligned(16))) float lds[Cfg::LDS];
    constexpr int ROWS = Cfg::ROWS, CT = Cfg::CT, KG = Cfg::KG, SL = Cfg::SL, AQ = ROWS / 8;
    constexpr int WPS = TERNARY ? 2 : 1;  // 32-bit weight words per column per step of 32 k
    using Acc = WavesAcc<Cfg>;

    const int tid = static_cast<int>(threadIdx.x);
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane / ROWS, col = lane % ROWS;  // k group and row / column of the lane's operands
    uint32_t ones;
    asm volatile("v_mov_b32 %0, 0x3f803f80" : "=v"(ones));

    // XCD x = blockIdx % 8 owns per_xcd consecutive tiles of an order that
    // walks group_r tile rows at a time
    const int t = (static_cast<int>(blockIdx.x) & 7) * per_xcd + (static_cast<int>(blockIdx.x) >> 3);
    if (t >= tiles_r * tiles_c) return;
    const int gr = t / (group_r * tiles_c);
    const int rows_here = min(group_r, tiles_r - gr * group_r);
    const int in = t - gr * group_r * tiles_c;
    const int r0 = (gr * group_r + in % rows_here) * ROWS;
    const int c0 = (in / rows_here) * Cfg::BC;

    // this wave's steps of 32 k
    const int all = (p.K + 31) / 32;
    const int per = (all + KG - 1) / KG;
    const int s0 = wave * per;
    const int n = max(0, min(per, all - s0));

    // A: lane -> rows lane / 8 + 8 i, 16-byte part lane % 8 of a row's 128
    // bytes per step; parts sit XOR-swizzled in the wave's LDS rows
    const float* a_base = p.A + static_cast<int64_t>(r0) * p.lda;
    const uint64_t a_bytes = (static_cast<uint64_t>(p.M - 1 - r0) * p.lda + p.K) * 4;
    const int lda = static_cast<int>(p.lda);
    const int a_voff = ((lane >> 3) * lda + (lane & 7) * 4) * 4;
    float* const stage = lds + wave * Cfg::STAGE;
    const int st_at = (lane >> 3) * 32 + (((lane & 7) ^ (lane >> 3)) * 4);
    // The k order inside a step is free as long as both operands share it.  A
    // lane's 8 weights of a slice are pairs of bits (codes) 16 bits apart in
    // a weight word, so one shift puts a pair at the sign bits of a dword of
    // two bf16: binary words hold 32 k, elements 2d and 2d + 1 are bits 4q + d
    // and 16 + 4q + d for q = slice * (lane groups) + lane group; ternary
    // words hold 16 k, codes 4q + d and 8 + 4q + d, q = 0 or 1.  The lane
    // therefore multiplies parts first(kk) and first(kk) + apart of its row.
    constexpr int apart = TERNARY ? 2 : 4;
    auto first = [&](int kk) {
        if constexpr (!TERNARY) return kk * 2 + g;         // ROWS 16: one slice, g = 0..3
        else return ROWS == 32 ? 4 * kk + g : 4 * (g >> 1) + (g & 1);
    };
    const float* part_at[AQ];
#pragma unroll
    for (int q = 0; q < AQ; ++q)
        part_at[q] = stage + col * 32 + (((first(q >> 1) + (q & 1) * apart) ^ (col & 7)) * 4);

    const uint8_t* b_base = p.packed + static_cast<int64_t>(c0) * p.col_bytes;
    const uint64_t b_bytes = c0 < p.N_pad ? static_cast<uint64_t>(p.N_pad - c0) * static_cast<uint64_t>(p.col_bytes) : 0;
    int b_voff[CT];
#pragma unroll
    for (int j = 0; j < CT; ++j) b_voff[j] = (j * ROWS + col) * static_cast<int>(p.col_bytes);

    f32x4_t areg[2][AQ];                     // A of two later steps, in flight
    f32x4_t frag[2][AQ];                     // lane's A values of this and the next step
    u32x4_t wreg[CT][WPS], wnext[CT][WPS];   // W words of this and the next four steps
    auto load_a = [&](f32x4_t (&v)[AQ], int i) {
        const uint64_t bytes = i < n ? a_bytes : 0;
        const __amdgpu_buffer_rsrc_t rs = buffer_range(a_base, bytes, static_cast<uint64_t>(s0 + i) * 128);
#pragma unroll
        for (int q = 0; q < AQ; ++q)
            v[q] = __builtin_bit_cast(
                f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rs, a_voff + q * 8 * lda * 4, 0, 0));
    };
    auto load_w = [&](u32x4_t (&w)[CT][WPS], int i) {
        const uint64_t bytes = i < n ? b_bytes : 0;
#pragma unroll
        for (int q = 0; q < WPS; ++q) {
            const __amdgpu_buffer_rsrc_t rs =
                buffer_range(b_base, bytes, static_cast<uint64_t>(s0 + i) * 4 * WPS + 16 * q);
#pragma unroll
            for (int j = 0; j < CT; ++j)
                w[j][q] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rs, b_voff[j], 0, 0));
        }
    };
    // a wave's LDS accesses execute in order, so one buffer serves all steps
    auto stage_a = [&](const f32x4_t (&v)[AQ], f32x4_t (&f)[AQ]) {
#pragma unroll
        for (int q = 0; q < AQ; ++q) *reinterpret_cast<f32x4_t*>(stage + st_at + q * 256) = v[q];
#pragma unroll
        for (int q = 0; q < AQ; ++q) f[q] = *reinterpret_cast<const f32x4_t*>(part_at[q]);
    };

    typename Acc::type acc[CT];
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
        for (int e = 0; e < Cfg::ACC; ++e) acc[j][e] = 0.0f;

    // the weights of slice kk of the step with words w[j][..] (step js of four)
    auto weights = [&](const u32x4_t (&w)[CT][WPS], int js, int kk, int j) {
        u32x4_t r;
        if constexpr (TERNARY) {
            // codes inverted: sign bit, "nonzero" bit = bf16 -2, +2 or 0
            const uint32_t w0 = w[j][js >> 1][2 * (js & 1)], w1 = w[j][js >> 1][2 * (js & 1) + 1];
            const uint32_t word = ROWS == 32 ? (kk ? w1 : w0) : (g & 2 ? w1 : w0);
            const uint32_t y = ~word >> (8 * (g & 1));
#pragma unroll
            for (int d = 0; d < 4; ++d) r[d] = (y << (14 - 2 * d)) & 0xC000C000u;
        } else {
            const uint32_t y = w[j][0][js] >> (4 * g);
#pragma unroll
            for (int d = 0; d < 4; ++d) r[d] = ((y << (15 - 8 * kk - d)) & 0x80008000u) | ones;
        }
        return r;
    };
    auto multiply = [&](f32x4_t (&f)[AQ], const u32x4_t (&w)[CT][WPS], int js, int i, auto masked) {
        if constexpr (decltype(masked)::value) {
#pragma unroll
            for (int q = 0; q < AQ; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if ((s0 + i) * 32 + (first(q >> 1) + (q & 1) * apart) * 4 + e >= p.K) f[q][e] = 0.0f;
        }
#pragma unroll
        for (int kk = 0; kk < SL; ++kk) {
            float x[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = f[2 * kk + (e & 1)][e >> 1];
            uint4 hi, mid, lo;
            split8(x, hi, mid, lo);
            const u32x4_t planes[3] = {{hi.x, hi.y, hi.z, hi.w}, {mid.x, mid.y, mid.z, mid.w}, {lo.x, lo.y, lo.z, lo.w}};
            u32x4_t bf[CT];
#pragma unroll
            for (int j = 0; j < CT; ++j) bf[j] = weights(w, js, kk, j);
#pragma unroll
            for (int pl = 0; pl < 3; ++pl)
#pragma unroll
                for (int j = 0; j < CT; ++j) acc[j] = Acc::mfma(planes[pl], bf[j], acc[j]);
        }
    };

    if (n > 0) {
        // step i stages step i + 1 from its registers, which then receive step
        // i + 3; the next four steps' W words are fetched as four steps start.
        // FULL: four steps that exist and lie below K, without a branch
        auto steps4 = [&](int i0, auto full) {
            constexpr bool FULL = decltype(full)::value;
            load_w(wnext, i0 + 4);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int i = i0 + j;
                if (FULL || i < n) {
                    stage_a(areg[(j + 1) & 1], frag[(j + 1) & 1]);
                    load_a(areg[(j + 1) & 1], i + 3);
                    multiply(frag[j & 1], wreg, j, i, std::integral_constant<bool, !FULL>{});
                }
                // without it the scheduler hoists later steps' splits and spills
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int j = 0; j < CT; ++j)
#pragma unroll
                for (int q = 0; q < WPS; ++q) wreg[j][q] = wnext[j][q];
        };
        load_a(areg[0], 0);
        load_w(wreg, 0);
        load_a(areg[1], 1);
        stage_a(areg[0], frag[0]);
        load_a(areg[0], 2);
        const int whole = min(n, p.K / 32 - s0);  // steps that lie below K
        int i = 0;
        for (; i + 4 <= whole; i += 4) steps4(i, std::true_type{});
        if (i < n) steps4(i, std::false_type{});
    }

    // sum the waves in wave order, P fragments at a time, and finish four
    // consecutive columns of a row per thread
    const bool bias_then_scale = (p.flags & TBN_EPI_BIAS_THEN_SCALE) != 0;
    const bool relu = (p.flags & TBN_EPI_RELU) != 0;
    constexpr int P = Cfg::P, PC = ROWS * P;
#pragma unroll
    for (int j0 = 0; j0 < CT; j0 += P) {
        __syncthreads();
#pragma unroll
        for (int j = 0; j < P; ++j)
#pragma unroll
            for (int e = 0; e < Cfg::ACC; ++e)
                lds[(wave * ROWS + Acc::row(e, lane)) * PC + j * ROWS + col] = acc[j0 + j][e];
        __syncthreads();
        for (int i = tid; i < ROWS * PC / 4; i += Cfg::NT) {
            const int r = i / (PC / 4), c = (i % (PC / 4)) * 4;
            const int m = r0 + r, nc0 = c0 + j0 * ROWS + c;
            if (m >= p.M || nc0 >= p.N) continue;
            f32x4_t s = *reinterpret_cast<const f32x4_t*>(lds + r * PC + c);
#pragma unroll
            for (int w = 1; w < KG; ++w) {
                const f32x4_t v = *reinterpret_cast<const f32x4_t*>(lds + (w * ROWS + r) * PC + c);
#pragma unroll
                for (int e = 0; e < 4; ++e) s[e] += v[e];
            }
            float* out = p.C + static_cast<int64_t>(m) * p.ldc + nc0;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int nc = min(nc0 + e, p.N - 1);
                const float mult = p.scale ? p.alpha * p.scale[nc] : p.alpha;
                const float b = p.bias ? p.bias[nc] : 0.0f;
                const float a = TERNARY ? s[e] * 0.5f : s[e];  // ternary sums are doubled
                float v = bias_then_scale ? (a + b) * mult : a * mult + b;
                if (p.cin) v += p.beta * (p.cin_1d ? p.cin[nc] : p.cin[static_cast<int64_t>(m) * p.N + nc]);
                if (relu) v = v > 0.0f ? v : 0.0f;
                if (nc0 + e < p.N) __builtin_nontemporal_store(v, out + e);
            }
        }
    }
}

template <class Cfg>
int launch_waves(const tbn_hip::WideGemmArgs& a, bool ternary, hipStream_t s) {
    const int tiles_r = static_cast<int>(tbn_hip::ceil_div(a.M, Cfg::ROWS));
    const int tiles_c = static_cast<int>(tbn_hip::ceil_div(a.N, Cfg::BC));
    TBN_REQUIRE(static_cast<int64_t>(tiles_r) * tiles_c < (1LL << 30), TBN_INVALID_SHAPE, "too many tiles");
    const int per_xcd = static_cast<int>(tbn_hip::ceil_div(static_cast<int64_t>(tiles_r) * tiles_c, 8));
    // rows of tiles walked together: the fewest A and W bytes per XCD
    int group = 1;
    double best = 0.0;
    for (int gr = 1; gr <= tiles_r; gr *= 2) {
        const double cols = std::min<double>(tiles_c, std::max(1.0, static_cast<double>(per_xcd) / gr));
        const double bytes = std::min(gr, per_xcd) * Cfg::ROWS * 4.0 * a.K + cols * Cfg::BC * static_cast<double>(a.col_bytes);
        if (gr == 1 || bytes < best) best = bytes, group = gr;
    }
    const dim3 grid(8u * static_cast<unsigned>(per_xcd));
    if (ternary)
        hipLaunchKernelGGL((gemm_waves_kernel<Cfg, true>), grid, dim3(Cfg::NT), 0, s, a, tiles_r, tiles_c, per_xcd, group);
    else
        hipLaunchKernelGGL((gemm_waves_kernel<Cfg, false>), grid, dim3(Cfg::NT), 0, s, a, tiles_r, tiles_c, per_xcd, group);
    return tbn_hip::check_launch("gemm_f32 (waves)");
}

}  // namespace

namespace tbn_hip {

// The variants by increasing tile.  M, N and K decide (so a product's bits
// depend on its shape alone); the aim is about one block per CU, since a second round
// of blocks costs as much as the first, and for K below 700 four waves instead
// of eight, whose sums are fewer to add.
//   * 32 x 128 (8 waves) up to one round of 256 tiles: 256 x 4096 x 4096 28.5
//     us against 35.0 for 32 x 64 and 34.8 for the staged 32 x 128 tile; with
//     4 waves, two blocks per CU, beyond: 2000^3 54.9 us against 68.3 with 8.
//   * 32 x 64 when it fits one round: 128 x 4096 x 4096 18.7 us against 21.1
//     for 16 x 64 and 25.1 for 32 x 128.
//   * 16 x 64: 64 x 4096 x 4096 13.4 us against 15.1 for 32 x 32.
//   * 16 x 32: 24 x 4096 x 4096 10.6 us against 14.1 for 16 x 16; for
//     K < 700 also in place of the two above: 600^3 7.1 us against 7.9 for 32 x 64.
//   * 16 x 16 for the rest: 1 x 4096 x 4096 9.0 us against 9.7 for 16 x 32.
int gemm_waves_plan(int M, int N, int K) {
    auto tiles = [&](int64_t r, int64_t c) { return ceil_div(M, r) * ceil_div(N, c); };
    const bool longer = K >= 700;
    const int64_t wide = tiles(32, 128);
    if (wide > 256) return 1;
    if (tiles(32, 64) > 256 && longer) return 0;
    if (tiles(32, 64) >= 160) return longer ? 2 : 4;
    if (tiles(16, 64) >= 160) return longer ? 3 : 4;
    if (tiles(16, 32) >= 160) return longer ? 5 : 4;
    return 6;
}

std::string gemm_waves_kernel_name(int plan, bool ternary) {
    static const char* cfg[] = {"32, 4, 8", "32, 4, 4", "32, 2, 8", "16, 4, 8", "16, 2, 4", "16, 2, 8", "16, 1, 8"};
    return std::string("gemm_waves_kernel<WavesCfg<") + cfg[plan] + ">, " + (ternary ? "true>" : "false>");
}

int gemm_waves(const WideGemmArgs& a, bool ternary, int plan, hipStream_t stream) {
    switch (plan) {
        case 0: return launch_waves<WavesCfg<32, 4, 8>>(a, ternary, stream);
        case 1: return launch_waves<WavesCfg<32, 4, 4>>(a, ternary, stream);
        case 2: return launch_waves<WavesCfg<32, 2, 8>>(a, ternary, stream);
        case 3: return launch_waves<WavesCfg<16, 4, 8>>(a, ternary, stream);
        case 4: return launch_waves<WavesCfg<16, 2, 4>>(a, ternary, stream);
        case 5: return launch_waves<WavesCfg<16, 2, 8>>(a, ternary, stream);
        default: return launch_waves<WavesCfg<16, 1, 8>>(a, ternary, stream);
    }
}

}  // namespace tbn_hip
