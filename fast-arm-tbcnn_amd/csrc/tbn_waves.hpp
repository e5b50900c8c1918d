// TBN-mode product with K split over the waves of a block (tbn_waves.hip).
#pragma once

#include "common.hpp"

namespace tbn_hip {

struct TbnWavesArgs {
    const float* A;
    int64_t lda;
    int M, N, K;
    const uint8_t* packed;  // BinaryMatrix columns, col_bytes = K_pad / 8 each
    int64_t col_bytes;
    int K_pad, N_pad;
    float scale, lo, hi;
    float* out;
    int64_t ldo;
};

// The variant for a shape, -1 where the two passes of tbn_mode.hip are faster.
int tbn_waves_plan(int M, int N);
int tbn_waves(const TbnWavesArgs& a, int plan, hipStream_t stream);

}  // namespace tbn_hip
