// What gemm.hip and gemm_bf16_pipe.hip agree on about a bf16 product whose A is k-contiguous.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace emi {

struct Bf16Plan {
  int shape;        // 0: the 256 x 256 ping-pong kernel of gemm.hip; otherwise a block shape of gemm_bf16_pipe.hip
  int splits;       // splits of K
};
Bf16Plan bf16_plan(int64_t M, int64_t N, int64_t K, int count, int sum, int trans_b);

int launch_bf16_pipe(hipStream_t st, const Bf16Plan& plan, int count, const void* const* A, const void* const* B, const void* const* R,
                     void* const* C, float* part, int M, int N, int K, int lda, int ldb, int64_t ldr, int64_t ldc, int vec_ok, int trans_b,
                     int sum);

}  // namespace emi
