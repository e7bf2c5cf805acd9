// fp32 GEMM on the bf16 matrix cores: launch parameters and host entry.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

namespace gptc {

// Row-major C (M x N) = op(A) op(B) (+ bias) (+ C).  A is (M x K) with rows
// of lda floats, or (K x M) when trans_a; B is (K x N), or (N x K) when
// trans_b.
struct SplitGemm {
    const float *A, *B;
    float *C;
    const float *bias;  // N values added to every row, or nullptr
    const float *add;   // (M x N) added to the product, rows of ldc (C itself to accumulate), or nullptr
    int M, N, K, lda, ldb, ldc;
    bool trans_a, trans_b;
};

// Whether the kernels of gemm_split.hip serve the problem (sizes and strides
// within their 32-bit tile offsets, a layout they are built for).
bool split_gemm_serves(const SplitGemm &g);

// Under graph capture the reduction stays whole: slices would take a block of the pool.
void launch_split_gemm(const SplitGemm &g, hipStream_t stream);

// C (M x N, rows of ldc) = the sum of the S products in part (M x N each, without gaps, one
// after the other; 16-byte aligned), in that order, (+ bias) (+ add, which may be C).
void launch_sum_slices(const float *part, const float *bias, const float *add, float *C, int M, int N, int ldc, int S,
                       hipStream_t stream);

}  // namespace gptc
