// What the fp32 product kernels share (gemm_f32.hip, gemm_f32_split.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace emi {

// Several products of one shape in one launch.  sum == 0: C[i] = op(A[i]) . op(B[i]) [+ R[i]];  sum == 1: every product
// is accumulated into the tile of C[0] (+ R[0]), pair after pair.
constexpr int kMaxF32Group = 48;
struct F32Group {
  const float* A[kMaxF32Group];
  const float* B[kMaxF32Group];
  const float* R[kMaxF32Group];
  float* C[kMaxF32Group];
  int count, sum;
};
struct F32Single {};

struct F32Call {
  const float *A, *B, *R;
  float* C;
  int M, N, K, lda, ldb;
  int64_t ldr, ldc;
  float* part;
  int splits;
  const F32Group* grp;       // nullptr: the single product of A and B
  int* planes;               // not null: splits stay planes in `part`, *planes of them (gemm_run)
};

// gemm.hip: adds `splits` planes [M, N] (+ R) into C in plane order
int launch_f32_splitk_reduce(hipStream_t st, const float* part, const float* R, float* C, int M, int N, int splits, int64_t ldr, int64_t ldc);

// gemm_f32_split.hip: shape 0: blocks of 128 x 128, 1: 128 x 64, 2: 64 x 64
int launch_f32_bf16x3(hipStream_t st, const F32Call& c, int shape, int trans_a, int trans_b);

}  // namespace emi
