// Tile, operand staging and inner loop shared by the fp32 GEMM
// (gemm_dense.hip) and the fp32 convolution (conv_dense.hip): chunks of k staged as
// fp32 in two LDS buffers, multiplied by v_mfma_f32_16x16x4_f32 with one
// chain of 4-value groups of k per wave (the order of the sum: gemm_dense.hip).
#pragma once

#include "mfma_core.hpp"

namespace tbnk {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
// 16-byte accesses of rows that are only 4-byte aligned (any K or N)
typedef float f32x4u_t __attribute__((ext_vector_type(4), aligned(4)));

template <int T_, int KC_>
struct DenseTile {
    static constexpr int T = T_;
    static constexpr int KC = KC_;                       // k per chunk
    static constexpr int PER = T * KC / 4 / 256;         // 16-byte items a thread stages per operand
    static constexpr int KPITCH = KC + 4;                // rows of contiguous k
    static constexpr int CPITCH = T == 16 ? 16 : T + 16; // rows of contiguous columns
    static constexpr int RPITCH = T + 4;                 // chain sums
    static constexpr int operand(bool kcont) { return kcont ? T * KPITCH : KC * CPITCH; }
    static_assert(T * KC % 1024 == 0 && 256 % (T / 4) == 0 && KC % 16 == 0, "whole 16-byte items per thread");
};

// One operand of a block: `row` is a row of op(A) or a column of op(B),
// element (row, k) at base[row * s_row + k * s_k] with s_k = 1 (KCONT) or
// s_row = 1; `stride` is the other one.  All loads are 16-byte buffer loads
// at offsets that are fixed per lane (the chunk moves the resource base,
// scalar work) over exactly the operand's bytes: the range check is per dword
// and takes any 4-byte alignment, so a value past the end of the matrix reads
// as zero.  One past the end of a row reads the next row's: of those, k >= K
// of a KCONT operand is zeroed as it is stored (the other operand's k >= K is
// past the matrix), and the others belong to outputs that are not stored.
template <class Tile, bool KCONT>
struct DenseOperand {
    static constexpr int T = Tile::T, KC = Tile::KC;
    const float* base;
    uint64_t bytes;
    int64_t stride;
    int voff[KCONT ? Tile::PER : 1];

    __device__ __forceinline__ DenseOperand(const float* b, int64_t st, int row0, int rows, int K) {
        const int tid = static_cast<int>(threadIdx.x);
        stride = st;
        base = b + row0 * (KCONT ? st : 1);
        bytes = static_cast<uint64_t>(KCONT ? (rows - 1 - row0) * st + K : (K - 1) * st + rows - row0) * 4;
        if constexpr (KCONT) {
#pragma unroll
            for (int j = 0; j < Tile::PER; ++j) {
                const int i = j * 256 + tid;
                voff[j] = ((i / (KC / 4)) * static_cast<int>(st) + (i % (KC / 4)) * 4) * 4;
            }
        } else {
            voff[0] = (tid / (T / 4)) * static_cast<int>(st * 4) + (tid % (T / 4)) * 16;
        }
    }
    __device__ __forceinline__ void load(f32x4_t (&v)[Tile::PER], int k0) const {
#pragma unroll
        for (int j = 0; j < Tile::PER; ++j) {
            const int k = KCONT ? k0 : k0 + j * (256 / (T / 4));
            const __amdgpu_buffer_rsrc_t rs =
                buffer_range(base, bytes, static_cast<uint64_t>(KCONT ? k : k * stride) * 4);
            v[j] = __builtin_bit_cast(f32x4_t,
                                      __builtin_amdgcn_raw_buffer_load_b128(rs, voff[KCONT ? j : 0], 0, 0));
        }
    }
    __device__ __forceinline__ void store(float* lds, f32x4_t (&v)[Tile::PER], int k0, int K) const {
        const int tid = static_cast<int>(threadIdx.x);
        if (KCONT && k0 + KC > K) {
#pragma unroll
            for (int j = 0; j < Tile::PER; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (k0 + ((j * 256 + tid) % (KC / 4)) * 4 + e >= K) v[j][e] = 0.0f;
        }
#pragma unroll
        for (int j = 0; j < Tile::PER; ++j) {
            const int i = j * 256 + tid;
            float* d = KCONT ? lds + (i / (KC / 4)) * Tile::KPITCH + (i % (KC / 4)) * 4
                             : lds + (i / (T / 4)) * Tile::CPITCH + (i % (T / 4)) * 4;
            *reinterpret_cast<f32x4_t*>(d) = v[j];
        }
    }
};

// One wave's chain over a staged chunk (operand A at buf, B at buf + kA):
// every step of the chunk, zeros past K included (fmaf(0, 0, acc) is acc); a
// step's operands are read during the step before.  A lane's operand element
// of row tile i is row i*16 + lane%16, k = 4 * chain + lane/16 (+ 16 per step).
template <class Tile, bool A_KCONT, bool B_KCONT>
__device__ __forceinline__ void dense_multiply(const float* buf, int chain, int lane,
                                               f32x4_t (&acc)[Tile::T / 16][Tile::T / 16]) {
    constexpr int F = Tile::T / 16, kA = Tile::operand(A_KCONT);
    const int kl = 4 * chain + (lane >> 4), rl = lane & 15;
    const int a_at = A_KCONT ? rl * Tile::KPITCH + kl : kl * Tile::CPITCH + rl;
    const int b_at = kA + (B_KCONT ? rl * Tile::KPITCH + kl : kl * Tile::CPITCH + rl);
    constexpr int a_tile = A_KCONT ? 16 * Tile::KPITCH : 16, a_step = A_KCONT ? 16 : 16 * Tile::CPITCH;
    constexpr int b_tile = B_KCONT ? 16 * Tile::KPITCH : 16, b_step = B_KCONT ? 16 : 16 * Tile::CPITCH;
    float a[2][F], b[2][F];
    auto read = [&](int s) {
#pragma unroll
        for (int i = 0; i < F; ++i) a[s & 1][i] = buf[a_at + i * a_tile + s * a_step];
#pragma unroll
        for (int j = 0; j < F; ++j) b[s & 1][j] = buf[b_at + j * b_tile + s * b_step];
    };
    read(0);
#pragma unroll
    for (int s = 0; s < Tile::KC / 16; ++s) {
        if (s + 1 < Tile::KC / 16) read(s + 1);
#pragma unroll
        for (int i = 0; i < F; ++i)
#pragma unroll
            for (int j = 0; j < F; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s & 1][i], b[s & 1][j], acc[i][j], 0, 0, 0);
    }
}

// The wave's chain of the tile into LDS (the chunk buffers are free after the
// last barrier): [chain][row][column], pitch RPITCH.
template <class Tile>
__device__ __forceinline__ void dense_put_chain(float* lds, int chain, int lane,
                                                const f32x4_t (&acc)[Tile::T / 16][Tile::T / 16]) {
    constexpr int F = Tile::T / 16;
#pragma unroll
    for (int i = 0; i < F; ++i)
#pragma unroll
        for (int j = 0; j < F; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                lds[(chain * Tile::T + i * 16 + 4 * (lane >> 4) + r) * Tile::RPITCH + j * 16 + (lane & 15)] =
                    acc[i][j][r];
}
// (chain 0 + chain 1) + (chain 2 + chain 3) of four consecutive columns
template <class Tile>
__device__ __forceinline__ f32x4_t dense_sum_chains(const float* lds, int row, int column) {
    f32x4_t s[4], y;
#pragma unroll
    for (int ch = 0; ch < 4; ++ch)
        s[ch] = *reinterpret_cast<const f32x4_t*>(lds + (ch * Tile::T + row) * Tile::RPITCH + column);
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = (s[0][e] + s[1][e]) + (s[2][e] + s[3][e]);
    return y;
}

}  // namespace tbnk
