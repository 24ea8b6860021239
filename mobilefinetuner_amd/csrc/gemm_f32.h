// fp32 matrix products on the bf16 matrix units (gemm_f32.hip): the products
// of the fp32 LM head and of the LoRA layer with an fp32 weight.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace mft {

// One term of a product: op(A) [M, K] times op(B) [K, N].  A is stored [M, K]
// with row stride lda, or [K, M] when ta; B [K, N] with row stride ldb, or
// [N, K] when tb.  A is multiplied by alpha.
struct GemmF32Term {
    const float* A;
    const float* B;
    int64_t lda, ldb, K;
    int ta, tb;
    float alpha;
};

// C[M, N] (row stride ldc) = sum of the terms (+ bias[n]) (+ C when add).
// terms[1].K = 0: one term.
struct GemmF32 {
    int64_t M, N, ldc;
    GemmF32Term terms[2];
    float* C;
    const float* bias;  // [N] or null
    int add;
    float* partial;     // workspace of gemm_f32_workspace bytes (may be null where that is 0)
};

// Workspace bytes: fp32 partial products where K is split across workgroups.
size_t gemm_f32_workspace(const GemmF32& g);
hipError_t launch_gemm_f32(const GemmF32& g, hipStream_t st);

}  // namespace mft
