// fp32 GEMM on the fp32 matrix instructions (gemm_dense.hip): products with
// more columns than a classifier head and a moderate K.
#pragma once

#include "common.hpp"

namespace tbn_hip {

struct DenseGemmArgs {
    const float* A;
    int64_t a_row, a_k;  // element (m, k) of op(A) at A[m*a_row + k*a_k]
    const float* B;
    int64_t b_k, b_col;  // element (k, n) of op(B) at B[k*b_k + n*b_col]
    int M, N, K;
    float alpha;
    const float* cin;    // null, [N] (cin_1d) or [M, N]
    int cin_1d;
    float beta;
    int flags;
    float* out;          // [M, N]
};

// From N and K only, so that a row's result never depends on how many rows
// the call has: every tile sums in the same order.  (A transposed A of more
// than 2^25 rows would pass the kernel's 32-bit lane offsets.)
inline bool gemm_dense_fits(int64_t M, int64_t N, int64_t K, bool transA) {
    return N > 64 && N <= 4096 && K >= 1 && K <= 4096 && (!transA || M <= (1 << 25));
}
int gemm_dense(const DenseGemmArgs& a, hipStream_t stream);

}  // namespace tbn_hip
