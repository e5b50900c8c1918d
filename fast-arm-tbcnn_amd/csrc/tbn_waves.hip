// TBN-mode product (qlinear_matmul_binary in the reference's own arithmetic,
// quantized_gemm_neon.cpp:160-243,380-430) in one launch, for products whose
// 256 x 256 tiles of tbn_mode.hip do not fill the chip.
//
// A block owns 16 or 32 rows of A (one fp4 matrix instruction) x 1 to 8
// fragments of as many columns; each of its 4 or 8 waves runs a contiguous
// part of K on the whole tile by itself, without a barrier.  It loads fp32
// rows (16 bytes a lane), turns them round through its own LDS rows so that a lane
// holds 32 values of its row, ternarizes them into the instruction's operand in
// registers, and expands 32 weight bits into the other with two instructions per
// dword.  The waves' sums, exact integers, are added through LDS.  No fp4 operand rows in
// memory, no workspace, one launch instead of two.
//
// What bounds it: vector instructions, about 5 per activation for the
// ternarization (a wider tile shares them among more columns), and latency
// below a few microseconds.
//
// Measured (kernel time, us; before = fp4 operand rows written to memory, then
// 256 x 256 tiles): 1 x 4096 x 4096 8.5 (28.9 before), 1 x 2073 x 131 7.4 (16.0),
// 64 x 4096 x 4096 12.2 (29.2), 512^3 5.7 (9.3), 1024^3 9.4 (12.4), 256 x
// 4096 x 4096 21.1 (30.9), 1733 x 3469 x 689 24.8 (36.0).
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "mfma_core.hpp"
#include "tbn_f4.hpp"
#include "tbn_waves.hpp"

namespace {

using namespace tbnk;

typedef float f32x4_t __attribute__((ext_vector_type(4)));

template <int ROWS_, int CT_, int KG_>
struct TbnWavesCfg {
    static constexpr int ROWS = ROWS_;       // rows of the tile: 32 (32x32x64 instructions) or 16 (16x16x128)
    static constexpr int CT = CT_;           // column fragments of ROWS columns
    static constexpr int KG = KG_;           // waves, each with a contiguous part of K
    static constexpr int NT = 64 * KG;
    static constexpr int BC = ROWS * CT;
    static constexpr int KSTEP = 2048 / ROWS;      // k per step: 32 per lane
    static constexpr int ROWPARTS = KSTEP / 4;     // 16-byte parts of a row per step
    static constexpr int ACC = ROWS * ROWS / 64;
    static constexpr int P = CT >= 2 ? 2 : 1;      // fragments summed per pass
    static constexpr int STAGE = 2048;             // floats a wave stages per step
    static constexpr int LDS = KG * STAGE;
    static_assert(P * ROWS * ROWS <= STAGE, "the sums fit the staging rows");
};

template <class Cfg>
struct TbnAcc;
template <int CT, int KG>
struct TbnAcc<TbnWavesCfg<32, CT, KG>> {
    using type = f32x16_t;
    static __device__ __forceinline__ type mfma(i32x4_t a, i32x4_t b, type c) { return mfma_f4(a, b, c); }
    static __device__ __forceinline__ int row(int e, int lane) { return 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3); }
};
template <int CT, int KG>
struct TbnAcc<TbnWavesCfg<16, CT, KG>> {
    using type = f32x4_t;
    static __device__ __forceinline__ type mfma(i32x4_t a, i32x4_t b, type c) {
        const i32x8_t a8 = {a[0], a[1], a[2], a[3], 0, 0, 0, 0};
        const i32x8_t b8 = {b[0], b[1], b[2], b[3], 0, 0, 0, 0};
        return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a8, b8, c, 4, 4, 0, 127, 0, 127);
    }
    static __device__ __forceinline__ int row(int e, int lane) { return 4 * (lane >> 4) + e; }
};

template <class Cfg>
__global__ void __launch_bounds__(Cfg::NT)
tbn_waves_kernel(tbn_hip::TbnWavesArgs p, int tiles_r, int tiles_c, int per_xcd, int group_r) {
    __shared__ __attribute__((aligned(16))) float lds[Cfg::LDS];
    constexpr int ROWS = Cfg::ROWS, CT = Cfg::CT, KG = Cfg::KG, KSTEP = Cfg::KSTEP, RP = Cfg::ROWPARTS;
    using Acc = TbnAcc<Cfg>;

    const int tid = static_cast<int>(threadIdx.x);
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane / ROWS, col = lane % ROWS;  // k group (32 k each) and row / column of the lane's operands

    // XCD x = blockIdx % 8 owns per_xcd consecutive tiles of an order that
    // walks group_r tile rows at a time
    const int t = (static_cast<int>(blockIdx.x) & 7) * per_xcd + (static_cast<int>(blockIdx.x) >> 3);
    if (t >= tiles_r * tiles_c) return;
    const int gr = t / (group_r * tiles_c);
    const int rows_here = min(group_r, tiles_r - gr * group_r);
    const int in = t - gr * group_r * tiles_c;
    const int r0 = (gr * group_r + in % rows_here) * ROWS;
    const int c0 = (in / rows_here) * Cfg::BC;

    // this wave's steps
    const int all = (p.K_pad + KSTEP - 1) / KSTEP;
    const int per = (all + KG - 1) / KG;
    const int s0 = wave * per;
    const int n = max(0, min(per, all - s0));

    // A: lane -> rows lane / RP + i * (64 / RP), 16-byte part lane % RP; parts
    // sit XOR-swizzled in the wave's LDS rows
    constexpr int RSTEP = 64 / RP;
    const float* a_base = p.A + static_cast<int64_t>(r0) * p.lda;
    const uint64_t a_bytes = (static_cast<uint64_t>(p.M - 1 - r0) * p.lda + p.K) * 4;
    const int lda = static_cast<int>(p.lda);
    const int a_row = lane / RP, a_part = lane % RP;
    const int a_voff = (a_row * lda + a_part * 4) * 4;
    float* const stage = lds + wave * Cfg::STAGE;
    const float* const frag_at = stage + col * KSTEP;

    const uint8_t* b_base = p.packed + static_cast<int64_t>(c0) * p.col_bytes;
    const uint64_t b_bytes = c0 < p.N_pad ? static_cast<uint64_t>(p.N_pad - c0) * static_cast<uint64_t>(p.col_bytes) : 0;
    int b_voff[CT];
#pragma unroll
    for (int j = 0; j < CT; ++j) b_voff[j] = (j * ROWS + col) * static_cast<int>(p.col_bytes) + 4 * g;

    f32x4_t areg[2][8];     // A of two later steps, in flight
    f32x4_t frag[2][8];     // lane's 32 A values of this and the next step
    uint32_t wreg[4][CT];   // W words of this and three later steps
    auto load_a = [&](f32x4_t (&v)[8], int i) {
        const __amdgpu_buffer_rsrc_t rs =
            buffer_range(a_base, i < n ? a_bytes : 0, static_cast<uint64_t>(s0 + i) * (KSTEP * 4));
#pragma unroll
        for (int q = 0; q < 8; ++q)
            v[q] = __builtin_bit_cast(
                f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rs, a_voff + q * RSTEP * lda * 4, 0, 0));
    };
    auto load_w = [&](uint32_t (&w)[CT], int i) {
        const __amdgpu_buffer_rsrc_t rs =
            buffer_range(b_base, i < n ? b_bytes : 0, static_cast<uint64_t>(s0 + i) * (KSTEP / 8));
#pragma unroll
        for (int j = 0; j < CT; ++j) w[j] = __builtin_amdgcn_raw_buffer_load_b32(rs, b_voff[j], 0, 0);
    };
    // a wave's LDS accesses execute in order, so one buffer serves all steps
    auto stage_a = [&](const f32x4_t (&v)[8], f32x4_t (&f)[8]) {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int r = a_row + q * RSTEP;
            *reinterpret_cast<f32x4_t*>(stage + r * KSTEP + ((a_part ^ (r & 7)) * 4)) = v[q];
        }
#pragma unroll
        for (int q = 0; q < 8; ++q)
            f[q] = *reinterpret_cast<const f32x4_t*>(frag_at + (((8 * g + q) ^ (col & 7)) * 4));
    };

    typename Acc::type acc[CT];
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
        for (int e = 0; e < Cfg::ACC; ++e) acc[j][e] = 0.0f;

    // The k order inside a lane's 32 is free as long as both operands share
    // it: nibble e of dword d is k = 4 e + d, so a weight dword is one shift and one
    // and-or of the 32 bits of its word (+1 = 0x2, -1 = 0xA).
    auto multiply = [&](f32x4_t (&f)[8], const uint32_t (&w)[CT], int i, auto masked) {
        const int k0 = (s0 + i) * KSTEP + 32 * g;
        if constexpr (decltype(masked)::value) {
            // the padding [K, K_pad) holds zeros, ternarized like any value
#pragma unroll
            for (int q = 0; q < 8; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (k0 + 4 * q + e >= p.K) f[q][e] = 0.0f;
        }
        i32x4_t a;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            uint32_t word = 0;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float v = f[e][d];
                const uint32_t hi = v > p.hi ? kF4Plus << (4 * e) : 0u;
                word |= v < p.lo ? kF4Minus << (4 * e) : hi;
            }
            a[d] = static_cast<int>(word);
        }
        if constexpr (decltype(masked)::value) {
            if (k0 >= p.K_pad) a = i32x4_t{0, 0, 0, 0};
        }
#pragma unroll
        for (int j = 0; j < CT; ++j) {
            i32x4_t b;
#pragma unroll
            for (int d = 0; d < 4; ++d) b[d] = static_cast<int>(((w[j] << (3 - d)) & 0x88888888u) | 0x22222222u);
            acc[j] = Acc::mfma(a, b, acc[j]);
        }
    };

    if (n > 0) {
        // step i stages step i + 1 from its registers, which then receive step
        // i + 3.  FULL: four steps that exist and lie below K, without a branch
        auto steps4 = [&](int i0, auto full) {
            constexpr bool FULL = decltype(full)::value;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int i = i0 + j;
                if (FULL || i < n) {
                    stage_a(areg[(j + 1) & 1], frag[(j + 1) & 1]);
                    load_a(areg[(j + 1) & 1], i + 3);
                    load_w(wreg[(j + 3) & 3], i + 3);
                    multiply(frag[j & 1], wreg[j], i, std::integral_constant<bool, !FULL>{});
                }
                // keeps later steps' values out of the registers
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        load_a(areg[0], 0);
        load_w(wreg[0], 0);
        load_a(areg[1], 1);
        load_w(wreg[1], 1);
        load_w(wreg[2], 2);
        stage_a(areg[0], frag[0]);
        load_a(areg[0], 2);
        const int whole = min(n, p.K / KSTEP - s0);  // steps that lie below K
        int i = 0;
        for (; i + 4 <= whole; i += 4) steps4(i, std::true_type{});
        for (; i < n; i += 4) steps4(i, std::false_type{});
    }

    // C is the sum of the waves (exact integers, any order), P fragments at a time
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
            for (int w = 1; w < KG; ++w) s += *reinterpret_cast<const f32x4_t*>(lds + (w * ROWS + r) * PC + c);
            float* out = p.out + static_cast<int64_t>(m) * p.ldo + nc0;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (nc0 + e < p.N) out[e] = s[e] * p.scale;
        }
    }
}

template <class Cfg>
int launch_tbn_waves(const tbn_hip::TbnWavesArgs& a, hipStream_t s) {
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
    hipLaunchKernelGGL(tbn_waves_kernel<Cfg>, dim3(8u * static_cast<unsigned>(per_xcd)), dim3(Cfg::NT), 0, s, a,
                       tiles_r, tiles_c, per_xcd, group);
    return tbn_hip::check_launch("qlinear_matmul_binary_tbn (waves)");
}

}  // namespace

namespace tbn_hip {

// The smallest tile whose count fits one round of blocks, one per CU (a second
// round costs as much as the first); -1 beyond, where the two passes of
// tbn_mode.hip ternarize every activation once.  Every product and sum is an
// exact integer, so the choice cannot change a result.
int tbn_waves_plan(int M, int N) {
    auto fits = [&](int64_t r, int64_t c) { return ceil_div(M, r) * ceil_div(N, c) <= 256; };
    if (fits(16, 16)) return 0;
    if (fits(16, 32)) return 1;
    if (fits(16, 64)) return 2;
    if (fits(32, 64)) return 3;
    if (fits(32, 128)) return 4;
    if (fits(32, 256)) return 5;
    return -1;
}

int tbn_waves(const TbnWavesArgs& a, int plan, hipStream_t stream) {
    switch (plan) {
        case 0: return launch_tbn_waves<TbnWavesCfg<16, 1, 8>>(a, stream);
        case 1: return launch_tbn_waves<TbnWavesCfg<16, 2, 8>>(a, stream);
        case 2: return launch_tbn_waves<TbnWavesCfg<16, 4, 8>>(a, stream);
        case 3: return launch_tbn_waves<TbnWavesCfg<32, 2, 8>>(a, stream);
        case 4: return launch_tbn_waves<TbnWavesCfg<32, 4, 4>>(a, stream);
        default: return launch_tbn_waves<TbnWavesCfg<32, 8, 4>>(a, stream);
    }
}

}  // namespace tbn_hip
