// The FP32 matrix-core product of the surrogate's training (mlp_gemm.hip).
#pragma once
#include "common.h"

namespace smk {

constexpr int kTrainWidth = 256;

// The pass's activation, rounded as sm_mlp_bias_silu rounds it (one division
// of z; a product with the sigmoid would round once more), and its derivative
// as sm_mlp_silu_backward.
__device__ inline float train_sigmoid(float z) { return 1.0f / (1.0f + __expf(-z)); }
__device__ inline float train_silu(float z) { return z / (1.0f + __expf(-z)); }

// What becomes of the product P = A B:
//   kEpiStore     C = alpha P + beta C
//   kEpiPart      C[split][m][n] = the product over the split's k range
//   kEpiSilu      C = P + vec[n], C2 = silu(C)           (ldc both)
//   kEpiSiluBack  C = P silu'(vec[m][n]) (vec with ldc), and the column sums
//                 of C over each row tile: C2[row tile][n] (N columns)
enum GemmEpi { kEpiStore = 0, kEpiPart = 1, kEpiSilu = 2, kEpiSiluBack = 3 };

struct GemmArgs {
  int64_t M = 0, N = 0, K = 0;
  const float *A = nullptr, *B = nullptr;
  int64_t lda = 0, ldb = 0;  // stride of the index that is not contiguous
  float *C = nullptr;
  int64_t ldc = 0;
  float *C2 = nullptr;
  const float *vec = nullptr;
  float alpha = 1.0f, beta = 0.0f;
  int nsplit = 1;  // kEpiPart: at most this many slices of k
};

// ak: A(m, k) = A[m lda + k], else A[m + k lda]; bk: B(k, n) = B[n ldb + k],
// else B[k ldb + n].  small: 64 x 64 tiles instead of 128 x 128 (few rows:
// more workgroups).  Takes what gemm32_takes accepts.
int gemm32(GemmEpi epi, bool ak, bool bk, const GemmArgs &g, bool small, hipStream_t s);
bool gemm32_takes(bool ak, bool bk, const GemmArgs &g);
// slices a kEpiPart product really has
int gemm32_splits(const GemmArgs &g);

}  // namespace smk
