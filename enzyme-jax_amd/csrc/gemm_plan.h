// Which blocks and how many splits of K a product runs on: bf16 products whose A is k-contiguous, and fp32 products.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace emi {

struct Bf16Plan {
  int shape;        // 0: the 256 x 256 ping-pong kernel of gemm.hip; otherwise a block shape of gemm_bf16_pipe.hip
  int splits;       // splits of K
  double us;        // the estimate
};
struct F32Plan {
  int shape;        // on the fp32 instructions 0: blocks of 64 x 64, 1: 32 x 32, 2: 128 x 128 (gemm_f32.hip); on the bf16
                    // instructions 3: 128 x 128, 4: 128 x 64, 5: 64 x 64 (gemm_f32_split.hip)
  int splits;
  double us;
};

// The best of the plans with at most `most` splits.  A shape that was chosen for its splits is a poor one without them, so
// a call plans with the splits that its workspace holds, and one without a workspace for a single pass over K (us, planned
// so | the blocks of the split plan in a single pass, B k-contiguous; bf16: 256 x 11008 x 4096 36 | 65, 300 x 4096 x 11008
// 60 | 104, 512 x 768 x 32000 89 | 238; fp32: 256 x 4096 x 11008 247 | 677, 512 x 768 x 32000 330 | 1955).
constexpr int64_t kAnySplits = 1 << 20;
Bf16Plan bf16_plan(int64_t M, int64_t N, int64_t K, int count, int sum, int trans_b, int64_t most);      // gemm_bf16_pipe.hip
int bf16_kernel(const Bf16Plan& plan, int64_t M, int64_t N, int64_t K, int count, int sum, int trans_b);
F32Plan f32_plan(int64_t M, int64_t N, int64_t K, int count, int sum, int trans_a, int64_t most);        // gemm_f32.hip

inline int64_t splits_held(const void* workspace, size_t bytes, int64_t M, int64_t N) {
  if (workspace == nullptr || (reinterpret_cast<uintptr_t>(workspace) & 15) != 0) return 1;
  const int64_t n = (int64_t)(bytes / ((size_t)M * N * sizeof(float)));
  return n < 1 ? 1 : n < kAnySplits ? n : kAnySplits;
}

// Splits of a sum of two long products: none where its tiles of 128 leave hardly a CU idle.  Two blocks on every CU are estimated
// at the rate of operands that the L2s still hold, which those of a long contraction are not: two of 1000 x 4096 x 4096, us,
// in two splits 85 (estimate 71), in one pass 84 (73), one by one 80; two of 1000 x 4096 x 11008 212 (163), one by one 178.
inline int64_t sum_splits(int64_t M, int64_t N, int64_t held) { return (M + 127) / 128 * ((N + 127) / 128) >= 192 ? 1 : held; }

// Whether several bf16 products of a shape are one launch at all: not where one alone has 256-tiles for most of the chip.
inline bool bf16_one_launch(int64_t M, int64_t N) { return (M + 255) / 256 * ((N + 255) / 256) < 192; }

// Whether products that can run as one launch, each in a single pass over K, run one by one: where each split over K is so
// much faster that together they are, by more than the estimates are off (`margin`: bf16 products of a few rows are
// estimated up to a third too fast, fp32 ones hardly).  A launch more each, and the gap before it.  us, one launch | one by one:
// bf16, B k-major, 2 x 16 x 4096 x 11008 55 | 38 (3 of them 59 | 62: as one); fp32, both k-major, 4 x 64 x 64 x 16384
// 119 | 41, 4 x 768 x 768 x 16384 791 | 635, 4 x 768 x 768 x 4096 198 | 210 (as one).
template <typename Plan> inline bool faster_one_by_one(const Plan& group, const Plan& one, int count, double margin) {
  return one.splits > 1 && margin * count * (one.us + 1.0) < group.us;
}

int launch_bf16_pipe(hipStream_t st, const Bf16Plan& plan, int count, const void* const* A, const void* const* B, const void* const* R,
                     void* const* C, float* part, int M, int N, int K, int lda, int ldb, int64_t ldr, int64_t ldc, int vec_ok, int trans_b,
                     int sum, int* planes);

// Lets a kernel have `bytes` of LDS, once (`configured`: one to a kernel; a race only repeats the call).
int reserve_lds(const void* kernel, int bytes, bool& configured);                                        // gemm.hip

// emi_gemm_ws and emi_gemm_grouped for a caller that adds the planes of a product split over K itself: with `planes` not null
// such a product leaves *planes fp32 planes [M, N] in the workspace, to be added in order and then to R, and C unwritten;
// *planes is 0 where C is complete.
int gemm_run(hipStream_t st, const void* A, const void* B, const void* R, void* C, void* workspace, size_t workspace_bytes, int64_t M,
             int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldr, int64_t ldc, int trans_a, int trans_b, int dtype, int* planes);
int gemm_grouped_run(hipStream_t st, int count, const void* const* A, const void* const* B, const void* const* R, void* const* C,
                     void* workspace, size_t workspace_bytes, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldr,
                     int64_t ldc, int trans_a, int trans_b, int sum, int dtype, int* planes);

// Products whose result goes through an elementwise operator, where that operator is worked out before the result leaves: what
// is left of a small model between two products are passes of 2 to 4 us over it.  Each returns -1 where the separate launches
// are the faster ones, or alone possible, and has then launched nothing.  A kTail... is the MODE of the product kernels.
enum { kTailNone, kTailGroup, kTailGated, kTailRotated, kTailAdjoint };
struct ProductTail {
  int mode;
  const void* B[3];            // gated: W3 in B[1];  rotated: the weights of up to three results
  void* C[3];                  // gated: h1, h3, g;  rotated: the results;  adjoint: dh1, dh3
  const float* table;          // rotated: results 0 .. rotated - 1 by the angle of row % seq
  int seq, head_dim, rotated, count;
  const void *h1, *h3;         // adjoint: the SwiGLU's operands; the product is the cotangent of its result
  const void *A1, *B1[3];      // rotated, unless A1 is null: each result is A B[i]^T + A1 B1[i]^T (a tangent's two products)
};
int launch_bf16_pipe_tail(hipStream_t st, const void* A, const void* B, const ProductTail& t, int M, int N, int K, int ldb, int trans_b);      // gemm_bf16_pipe.hip
int launch_f32_tail(hipStream_t st, const void* A, const void* B, const ProductTail& t, int64_t M, int64_t N, int64_t K, int64_t ldb, int trans_b);      // gemm_f32.hip
int gemm_tail(hipStream_t st, const void* A, const void* B, const ProductTail& t, int64_t M, int64_t N, int64_t K, int64_t ldb, int trans_b, int dtype);   // gemm.hip

}  // namespace emi
