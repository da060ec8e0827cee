// RMSNorm adjoints whose dgamma is summed later, for drivers that run several of them (elementwise.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace emi {

constexpr int kMaxColsums = 96;
struct Colsums {                     // dgamma of one adjoint each: `rows` fp32 partial rows of `dim`
  const float* part[kMaxColsums];
  void* out[kMaxColsums];
};

// Partial rows that emi_rmsnorm_bwd leaves for [rows, dim], and whether one pass sums them (dim a multiple of 8 up to 8192).
int64_t rmsnorm_partial_rows(int64_t rows, int64_t dim);
bool rmsnorm_one_pass(int64_t dim);

// emi_rmsnorm_bwd without the column sum: dgamma's partial rows stay in `part`.  With dy_planes > 0, dy is the sum of that many
// fp32 planes [rows, dim], in order, rounded to the storage type.
int launch_rmsnorm_bwd_rows(hipStream_t st, const void* x, const void* gamma, const void* dy, int dy_planes, const void* dx_add, void* dx,
                            float* part, int64_t rows, int64_t dim, float eps, int dtype);
// x = the sum of `count` fp32 planes [rows, dim], in order, + r, rounded to the storage type; y = rmsnorm(x) gamma.
int launch_rmsnorm_fwd_planes(hipStream_t st, const float* planes, int count, const void* r, const void* gamma, void* x, void* y,
                              int64_t rows, int64_t dim, float eps, int dtype);
// out[i] = column sums of part[i], i < count, in one launch.
int launch_colsums(hipStream_t st, const Colsums& c, int count, int64_t part_rows, int64_t dim, int dtype);

}  // namespace emi
