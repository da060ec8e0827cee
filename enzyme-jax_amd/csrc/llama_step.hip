// The reference's own program as one call each way: a decoder step of one token through all layers (test/llama.py:35-238)
// and its reverse (every weight and both caches).
//
// Small models are a chain of launches, each as long as its latencies (a few us), and large ones are bound by the weights,
// which are read once (and, in reverse, read and written once).  Both want the fewest kernels: what lies between two
// matrix-vector products - RMSNorm, the rotation, SwiGLU, residuals, the new cache row - is done where its operand is
// loaded or its result leaves, and the cache is not copied to append a row to it.
//   forward, per layer:  norm + wq,wk,wv + rotation | attention over cache and own row (| combine) | wo + residual |
//                        norm + w1,w3 + SwiGLU | w2 + residual;  with a short cache attention + wo + residual are one
//   reverse, per layer:  w2^T dy and dw2 | SwiGLU' | w1^T dh1 + w3^T dh3 and dw1, dw3 | norm' (+ residual) |
//                        wo^T dy and dwo | sum | attention' (|) dq, inverse rotation | wq^T dq + ... and dwq, dwk, dwv | norm'
// The forward call leaves what the reverse one needs in `saved`.
// Measured against the same step operator by operator (us): dim 288, 6 layers, fp32: forward 1071 -> 100 (99 launches ->
// 25), with the reverse from StableHLO text at position 255 4042 -> 412 (289 launches -> 86); dim 4096, 2 layers, bf16,
// 4096 keys: forward 370 -> 211 (4.5 TB/s over weights and cache; 31 launches and two copies of each cache before).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "emi_device.h"

namespace emi {

int launch_skinny(hipStream_t st, const void* A, const void* B, const void* R, void* C, void* workspace, size_t workspace_bytes,
                  int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldr, int64_t ldc, int trans_a, int trans_b,
                  int dtype);                                                                                // gemm_skinny.hip
int launch_llama_step_attn_fwd(hipStream_t st, const void* q, const void* k_cache, const void* v_cache, const void* k_tail,
                               const void* v_tail, void* o, float* lse, float* part, int heads, int pos, int head_dim, int keys_per_block,
                               float scale, int dtype);                                                      // attention_step.hip
int launch_llama_step_attn_bwd(hipStream_t st, const void* q, const void* k_cache, const void* v_cache, const void* k_tail,
                               const void* v_tail, const void* o, const float* lse, const void* d_o, void* dk_cache, void* dv_cache,
                               void* dk_tail, void* dv_tail, float* part, const float* table, int table_pairs, float* fq, float* fk, float* fv,
                               int heads, int pos, int head_dim, int keys_per_block, float scale, int dtype);

namespace {

typedef float f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float block_sum_f32(float v, float* scratch) {          // scratch: one float per wavefront
  v = wave_sum(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = v;
  __syncthreads();
  float s = 0.f;
  for (int w = 0; w < (int)(blockDim.x >> 6); w++) s += scratch[w];
  return s;
}

template <typename T> __device__ __forceinline__ float round_to(float v) { return to_f32(from_f32<T>(v)); }
template <typename T> __device__ __forceinline__ float normed(float x, float gamma, float rs) { return round_to<T>(gamma * (x * rs)); }

// ---------------------------------------------------------------------------
// forward: products of a normalised vector
// ---------------------------------------------------------------------------
// A wavefront owns two rows at a time: MODE 0, rows 2p and 2p + 1 of [w0; w1; w2] (q, k, v: a rotation pair of q or k);
// MODE 1, row p of w0 and of w1 (h1, h3 of the SwiGLU); MODE 2, rows 2p and 2p + 1 of w0 (wo) times the attention's result,
// which each block works out for itself (step_attention).  The rows stream through in batches of UN 16-byte pieces per lane,
// the next pair's first batch requested while the current one is summed, and the first pair's before the block normalises
// the vector: each block keeps gamma x / rms(x) in LDS (the two halves of an eight-element piece apart, so that a
// lane's reads of 16 bytes do not collide).
template <typename T> struct NormGemv {
  const T *x, *gamma;    // MODE 2: x is the residual
  const T* w[3];
  T* y[3];               // MODE 0: q, k, v;  MODE 1: h1, h3, g;  MODE 2: x + w0 att
  float* rms;            // 1 / rms(x), for the adjoint
  const float2* table;   // MODE 0: (cos, sin) of pair i at i % table_pairs
  int N, K, table_pairs;
  float eps;
  // MODE 2: the attention whose result the vector is
  const T *q, *k_cache, *v_cache, *k_own, *v_own;
  T* att;
  float* lse;
  int heads, head_dim, keys;
  float scale;
};

// att of one query over a short cache and its own row, into the vector's LDS image: a row of 16 lanes holds a head (one
// 16-byte piece a lane), 16 heads at a time, kStepKeys keys requested together.  Each such round costs every block one
// latency of the L2, about 1.2 us a layer; the launch it saves costs 4 us where the host is the bound and 3 where the GPU is.
// So it is taken up to two rounds (StepDims::short_cache).  Forward, separate -> together, us (6 layers at dim 288 and 768,
// else 2):                  1 round            2 rounds           4 rounds
//   f32  288,  6 heads      126 -> 100         123 -> 103         124 -> 106
//   f32  768, 12 heads      134 -> 117         134 -> 124         134 -> 138
//   bf16 2048, 16 heads    82.5 -> 76.8       82.4 -> 79.9       82.7 -> 86.3
//   bf16 4096, 32 heads                      168.5 -> 165.5     168.5 -> 174.1
constexpr int kStepKeys = 8, kStepRounds = 2;
template <typename T> __device__ __forceinline__ void step_attention(const NormGemv<T>& a, float* xs, int pieces, bool store) {
  using Raw = typename ChunkCached<T>::Raw;
  constexpr int V = ChunkCached<T>::N;
  const int l16 = threadIdx.x & 15;
  const bool mine = l16 * V < a.head_dim;
  for (int h = threadIdx.x >> 4; h < a.heads; h += 16) {
    const int at = h * a.head_dim + l16 * V;
    float qf[V], acc[V];
#pragma unroll
    for (int e = 0; e < V; e++) qf[e] = acc[e] = 0.f;
    if (mine) ChunkCached<T>::load(a.q + at, qf);
    float mx = -INFINITY, sum = 0.f;
    for (int s0 = 0; s0 < a.keys; s0 += kStepKeys) {
      Raw kr[kStepKeys], vr[kStepKeys];
#pragma unroll
      for (int u = 0; u < kStepKeys; u++) {
        const int s = s0 + u;
        kr[u] = vr[u] = Raw{};
        if (mine && s < a.keys) {
          const bool own = s == a.keys - 1;
          kr[u] = ChunkCached<T>::load_raw((own ? a.k_own : a.k_cache + (int64_t)s * a.K) + at);
          vr[u] = ChunkCached<T>::load_raw((own ? a.v_own : a.v_cache + (int64_t)s * a.K) + at);
        }
      }
      float sc[kStepKeys], nm = mx;
#pragma unroll
      for (int u = 0; u < kStepKeys; u++) {
        float kf[V], dot = 0.f;
        ChunkCached<T>::unpack(kr[u], kf);
#pragma unroll
        for (int e = 0; e < V; e++) dot = fmaf(qf[e], kf[e], dot);
        dot = row16_sum(dot);
        sc[u] = s0 + u < a.keys ? dot * a.scale : -INFINITY;
        nm = fmaxf(nm, sc[u]);
      }
      const float alpha = mx == -INFINITY ? 0.f : __expf(mx - nm);
      sum *= alpha;
#pragma unroll
      for (int e = 0; e < V; e++) acc[e] *= alpha;
      mx = nm;
#pragma unroll
      for (int u = 0; u < kStepKeys; u++) {
        const float p = sc[u] == -INFINITY ? 0.f : __expf(sc[u] - mx);
        sum += p;
        float vf[V];
        ChunkCached<T>::unpack(vr[u], vf);
#pragma unroll
        for (int e = 0; e < V; e++) acc[e] = fmaf(p, vf[e], acc[e]);
      }
    }
    const float inv = 1.0f / sum;
    if (mine) {
#pragma unroll
      for (int e = 0; e < V; e++) acc[e] = round_to<T>(acc[e] * inv);
      if (store) ChunkCached<T>::store(a.att + at, acc);
#pragma unroll
      for (int g = 0; g < V / 4; g++)
        *reinterpret_cast<f4*>(xs + (g * pieces + at / V) * 4) = f4{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
    }
    if (store && l16 == 0) a.lse[h] = mx + __logf(sum);
  }
}

template <typename T, int MODE, int UN, bool WHOLE>       // WHOLE: rows are whole batches
__global__ __launch_bounds__(256) void step_norm_gemv_kernel(NormGemv<T> a) {
  using Raw = typename ChunkCached<T>::Raw;
  constexpr int V = ChunkCached<T>::N, BATCH = 64 * V * UN;
  extern __shared__ __attribute__((aligned(16))) float xs[];          // [V / 4][Kp / V][4], Kp = K rounded up to whole batches
  __shared__ float scratch[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nb = (a.K + BATCH - 1) / BATCH, pieces = nb * 64 * UN;     // pieces of the padded vector
  const int P = MODE == 0 ? 3 * a.N / 2 : MODE == 1 ? a.N : a.N / 2;
  auto rows = [&](int p, const T*& r0, const T*& r1) {
    if constexpr (MODE == 2) {
      r0 = a.w[0] + (int64_t)(2 * p) * a.K;
      r1 = r0 + a.K;
    } else if constexpr (MODE == 0) {
      const int m = 2 * p / a.N;
      r0 = (m == 0 ? a.w[0] : m == 1 ? a.w[1] : a.w[2]) + (int64_t)(2 * p - m * a.N) * a.K;
      r1 = r0 + a.K;
    } else {
      r0 = a.w[0] + (int64_t)p * a.K;
      r1 = a.w[1] + (int64_t)p * a.K;
    }
  };
  // unconditional: a piece past the row re-reads its start and is dropped when it is summed (a zero of the vector alone
  // would make a NaN of an infinite weight there)
  auto issue = [&](const T* r0, const T* r1, int b, Raw(&x0)[UN], Raw(&x1)[UN]) {
#pragma unroll
    for (int u = 0; u < UN; u++) {
      const int k = b * BATCH + (u * 64 + lane) * V, kk = k < a.K ? k : 0;
      x0[u] = Chunk<T>::load_raw(r0 + kk);
      x1[u] = Chunk<T>::load_raw(r1 + kk);
    }
  };
  const int p0 = blockIdx.x * 4 + wave, stride = gridDim.x * 4;
  const T *r0 = nullptr, *r1 = nullptr;
  Raw c0[UN], c1[UN], n0[UN], n1[UN];
  if (p0 < P) {
    rows(p0, r0, r1);
    issue(r0, r1, 0, c0, c1);
  }
  // the vector: the attention's or the norm's result, rounded to T as the operator-by-operator form stores it
  if constexpr (MODE == 2) {
    step_attention<T>(a, xs, pieces, blockIdx.x == 0);
    for (int c = a.K / V + threadIdx.x; c < pieces; c += 256)
#pragma unroll
      for (int h = 0; h < V / 4; h++) *reinterpret_cast<f4*>(xs + (h * pieces + c) * 4) = f4{0.f, 0.f, 0.f, 0.f};
  } else {
    float ss = 0.f;
    for (int c = threadIdx.x; c * V < a.K; c += 256) {
      float xv[V];
      ChunkCached<T>::load(a.x + c * V, xv);
#pragma unroll
      for (int e = 0; e < V; e++) ss = fmaf(xv[e], xv[e], ss);
    }
    const float rs = 1.0f / sqrtf(block_sum_f32(ss, scratch) / a.K + a.eps);
    if (blockIdx.x == 0 && threadIdx.x == 0) *a.rms = rs;
    for (int c = threadIdx.x; c < pieces; c += 256) {
      float o[V];
#pragma unroll
      for (int e = 0; e < V; e++) o[e] = 0.f;
      if (c * V < a.K) {
        float xv[V], gv[V];
        ChunkCached<T>::load(a.x + c * V, xv);
        ChunkCached<T>::load(a.gamma + c * V, gv);
#pragma unroll
        for (int e = 0; e < V; e++) o[e] = normed<T>(xv[e], gv[e], rs);
      }
#pragma unroll
      for (int h = 0; h < V / 4; h++) *reinterpret_cast<f4*>(xs + (h * pieces + c) * 4) = f4{o[4 * h], o[4 * h + 1], o[4 * h + 2], o[4 * h + 3]};
    }
  }
  __syncthreads();

  float s0 = 0.f, s1 = 0.f;
  auto consume = [&](int b, const Raw(&x0)[UN], const Raw(&x1)[UN]) {
#pragma unroll
    for (int u = 0; u < UN; u++) {
      float w0[V], w1[V];
      const int c = b * 64 * UN + u * 64 + lane;
      const Raw none{};
      const bool in_row = WHOLE || c * V < a.K;
      ChunkCached<T>::unpack(in_row ? x0[u] : none, w0);
      ChunkCached<T>::unpack(in_row ? x1[u] : none, w1);
#pragma unroll
      for (int h = 0; h < V / 4; h++) {
        const f4 xv = *reinterpret_cast<const f4*>(xs + (h * pieces + c) * 4);
#pragma unroll
        for (int e = 0; e < 4; e++) {
          s0 = fmaf(w0[4 * h + e], xv[e], s0);
          s1 = fmaf(w1[4 * h + e], xv[e], s1);
        }
      }
    }
  };
  auto finish = [&](int p) {
    if constexpr (MODE == 2) {                             // rows and residual in fp32, rounded once
      const float v0 = wave_sum(s0), v1 = wave_sum(s1);
      s0 = s1 = 0.f;
      if (lane == 0) {
        a.y[0][2 * p] = from_f32<T>(v0 + to_f32(a.x[2 * p]));
        a.y[0][2 * p + 1] = from_f32<T>(v1 + to_f32(a.x[2 * p + 1]));
      }
      return;
    }
    const float v0 = round_to<T>(wave_sum(s0)), v1 = round_to<T>(wave_sum(s1));
    s0 = s1 = 0.f;
    if (lane != 0) return;
    if constexpr (MODE == 0) {
      const int m = 2 * p / a.N, r = 2 * p - m * a.N;
      T* y = (m == 0 ? a.y[0] : m == 1 ? a.y[1] : a.y[2]) + r;
      if (m < 2) {
        const float2 t = a.table[(r >> 1) % a.table_pairs];
        y[0] = from_f32<T>(t.x * v0 - t.y * v1);
        y[1] = from_f32<T>(t.y * v0 + t.x * v1);
      } else {
        y[0] = from_f32<T>(v0);
        y[1] = from_f32<T>(v1);
      }
    } else {
      a.y[0][p] = from_f32<T>(v0);
      a.y[1][p] = from_f32<T>(v1);
      a.y[2][p] = from_f32<T>(emi_swiglu(v0, v1));
    }
  };
  // batches of this wavefront's pairs in one sequence, two register sets
  int p = p0, b = 0;
  auto next = [&](int& np, int& nbat, const T*& q0, const T*& q1) {
    np = p;
    nbat = b + 1;
    q0 = r0;
    q1 = r1;
    if (nbat == nb) {
      nbat = 0;
      np += stride;
      if (np < P) rows(np, q0, q1);
    }
  };
  while (p < P) {
    int np, nbat;
    const T *q0, *q1;
    next(np, nbat, q0, q1);
    if (np < P) issue(q0, q1, nbat, n0, n1);
    consume(b, c0, c1);
    if (b == nb - 1) finish(p);
    p = np, b = nbat, r0 = q0, r1 = q1;
    if (p >= P) break;
    next(np, nbat, q0, q1);
    if (np < P) issue(q0, q1, nbat, c0, c1);
    consume(b, n0, n1);
    if (b == nb - 1) finish(p);
    p = np, b = nbat, r0 = q0, r1 = q1;
  }
}

template <typename T, int MODE> int launch_norm_gemv(hipStream_t st, const NormGemv<T>& a) {
  constexpr int V = ChunkCached<T>::N;
  const int P = MODE == 0 ? 3 * a.N / 2 : MODE == 1 ? a.N : a.N / 2;
  // two blocks a CU: each normalises the vector once for all its pairs
  const unsigned grid = (unsigned)((P + 3) / 4 < 512 ? (P + 3) / 4 : 512);
#define EMI_NORM_GEMV(UN)                                                                                                      \
  do {                                                                                                                         \
    constexpr int batch = 64 * V * UN;                                                                                         \
    const size_t lds = (size_t)((a.K + batch - 1) / batch) * batch * sizeof(float);                                            \
    if (a.K % batch == 0) hipLaunchKernelGGL((step_norm_gemv_kernel<T, MODE, UN, true>), dim3(grid), dim3(256), lds, st, a);                   \
    else hipLaunchKernelGGL((step_norm_gemv_kernel<T, MODE, UN, false>), dim3(grid), dim3(256), lds, st, a);                                   \
  } while (0)
  if (a.K <= 64 * V * 2) EMI_NORM_GEMV(2);
  else EMI_NORM_GEMV(8);
#undef EMI_NORM_GEMV
  EMI_CHECK_LAUNCH("emi_llama_step(norm + products)");
  return EMI_OK;
}

// y = gamma x / rms(x) of one vector, and 1 / rms.
template <typename T>
__global__ __launch_bounds__(1024) void step_norm_kernel(const T* __restrict__ x, const T* __restrict__ gamma, T* __restrict__ y,
                                                         float* __restrict__ rms, int D, float eps) {
  __shared__ float scratch[16];
  float ss = 0.f;
  for (int i = threadIdx.x; i < D; i += 1024) {
    const float v = to_f32(x[i]);
    ss = fmaf(v, v, ss);
  }
  const float rs = 1.0f / sqrtf(block_sum_f32(ss, scratch) / D + eps);
  if (threadIdx.x == 0) *rms = rs;
  for (int i = threadIdx.x; i < D; i += 1024) y[i] = from_f32<T>(to_f32(gamma[i]) * (to_f32(x[i]) * rs));
}

// ---------------------------------------------------------------------------
// reverse: W^T dy and dW = dy x^T of up to three matrices [K, N] that share x (and the cotangent of x)
// ---------------------------------------------------------------------------
// Every row of a matrix is read once (for the cotangent of x) while its gradient's row is written; HBM-bound on both.  A
// thread owns one 16-byte piece of columns; a block's row lanes (as many as its columns leave) take the rows of a band in
// turn, two register sets of UN rows in flight, and meet through LDS.  The bands' sums [bands][N] go to `part` in fp32.
template <typename T> struct Adjoint {
  const T* w[3];
  T* dw[3];
  const float* dy[3];
  const T *x, *gamma;      // the products' operand: x, or with gamma the normalised gamma x rms
  const float* rms;
  float* part;
  int count, K, N, rows_per_band;
};

template <typename T, bool STREAM>
__global__ __launch_bounds__(256) void step_adjoint_kernel(Adjoint<T> a) {
  using Raw = typename ChunkCached<T>::Raw;
  constexpr int V = ChunkCached<T>::N, UN = 8;
  __shared__ float red[256][V + 1];
  const int pieces = a.N / V;
  const int width = pieces < 256 ? pieces : 256, lanes = 256 / width;       // columns of a block, row lanes
  const int rl = threadIdx.x / width, cl = threadIdx.x % width;
  const int piece = blockIdx.x * width + cl, n = piece * V;
  const bool live = rl < lanes && piece < pieces;
  const int total = a.count * a.K;
  const int r_begin = blockIdx.y * a.rows_per_band, r_end = r_begin + a.rows_per_band < total ? r_begin + a.rows_per_band : total;
  float acc[V], xv[V];
#pragma unroll
  for (int e = 0; e < V; e++) acc[e] = xv[e] = 0.f;
  if (live) {
    ChunkCached<T>::load(a.x + n, xv);
    if (a.gamma != nullptr) {
      float gv[V];
      ChunkCached<T>::load(a.gamma + n, gv);
      const float rs = *a.rms;
#pragma unroll
      for (int e = 0; e < V; e++) xv[e] = normed<T>(xv[e], gv[e], rs);
    }
    auto matrix = [&](int r) { return a.count == 1 ? 0 : r / a.K; };
    auto pick = [](auto&& p, int m) { return m == 0 ? p[0] : m == 1 ? p[1] : p[2]; };
    auto issue = [&](int r0, Raw(&w)[UN], float(&d)[UN]) {
#pragma unroll
      for (int u = 0; u < UN; u++) {
        const int r = r0 + u * lanes < r_end ? r0 + u * lanes : r_end - 1;            // past the band: its last row, unused
        const int m = matrix(r), k = r - m * a.K;
        w[u] = Chunk<T>::load_raw(pick(a.w, m) + (int64_t)k * a.N + n);
        d[u] = pick(a.dy, m)[k];
      }
    };
    auto consume = [&](int r0, const Raw(&w)[UN], const float(&d)[UN]) {
#pragma unroll
      for (int u = 0; u < UN; u++) {
        const int r = r0 + u * lanes;
        if (r < r_end) {
          const int m = matrix(r), k = r - m * a.K;
          float wv[V], o[V];
          ChunkCached<T>::unpack(w[u], wv);
#pragma unroll
          for (int e = 0; e < V; e++) {
            acc[e] = fmaf(d[u], wv[e], acc[e]);
            o[e] = d[u] * xv[e];
          }
          T* dst = pick(a.dw, m) + (int64_t)k * a.N + n;
          if constexpr (STREAM) Chunk<T>::store(dst, o);
          else ChunkCached<T>::store(dst, o);
        }
      }
    };
    Raw w0[UN], w1[UN];
    float d0[UN], d1[UN];
    int r = r_begin + rl;
    if (r < r_end) issue(r, w0, d0);
    while (r < r_end) {
      const int r1 = r + UN * lanes;
      if (r1 < r_end) issue(r1, w1, d1);
      consume(r, w0, d0);
      if (r1 >= r_end) break;
      r = r1 + UN * lanes;
      if (r < r_end) issue(r, w0, d0);
      consume(r1, w1, d1);
    }
  }
  if (lanes > 1) {
#pragma unroll
    for (int e = 0; e < V; e++) red[threadIdx.x][e] = acc[e];
    __syncthreads();
    if (rl == 0 && live) {
      for (int l = 1; l < lanes; l++)
#pragma unroll
        for (int e = 0; e < V; e++) acc[e] += red[l * width + cl][e];
    }
  }
  if (rl == 0 && live) {
    float* dst = a.part + (int64_t)blockIdx.y * a.N + n;
#pragma unroll
    for (int e = 0; e < V; e += 4) *reinterpret_cast<f4*>(dst + e) = f4{acc[e], acc[e + 1], acc[e + 2], acc[e + 3]};
  }
}

// Bands of rows: about two blocks per CU where there are rows enough, at least two rows per row lane.
template <typename T> int adjoint_bands(int count, int K, int N) {
  constexpr int V = ChunkCached<T>::N;
  const int pieces = N / V, width = pieces < 256 ? pieces : 256, lanes = 256 / width, cols = (pieces + width - 1) / width;
  int bands = (512 + cols - 1) / cols;
  const int most = (count * K + 2 * lanes - 1) / (2 * lanes);
  if (bands > most) bands = most;
  if (bands > 96 && N <= 1024) bands = 96;           // short vectors: the bands are summed by one block (step_norm_adjoint_kernel)
  return bands < 1 ? 1 : bands;
}

template <typename T> int launch_adjoint(hipStream_t st, Adjoint<T> a, int* bands) {
  constexpr int V = ChunkCached<T>::N;
  const int pieces = a.N / V, width = pieces < 256 ? pieces : 256;
  const int want = adjoint_bands<T>(a.count, a.K, a.N), total = a.count * a.K;
  a.rows_per_band = (total + want - 1) / want;
  *bands = (total + a.rows_per_band - 1) / a.rows_per_band;
  const dim3 grid((unsigned)((pieces + width - 1) / width), (unsigned)*bands);
  if ((size_t)total * a.N * sizeof(T) > ((size_t)32 << 20))
    hipLaunchKernelGGL((step_adjoint_kernel<T, true>), grid, dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((step_adjoint_kernel<T, false>), grid, dim3(256), 0, st, a);
  EMI_CHECK_LAUNCH("emi_llama_step(adjoint products)");
  return EMI_OK;
}

// In pairs: the bands' sums are longer than the chains within them (768 columns: 96 bands of 43 rows), and added one by
// one they decided the error.
__device__ __forceinline__ float sum8(const float (&t)[8]) { return ((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7])); }

// The sum over the bands of 16 columns per block: 16 band lanes with up to eight loads in flight each, met through LDS in
// order.  The result is valid in threads 0 .. 15.
__device__ __forceinline__ float sum_bands16(const float* __restrict__ part, int bands, int N, int n, float (*red)[16]) {
  const int col = threadIdx.x & 15, bl = threadIdx.x >> 4;
  float v = 0.f;
  if (n < N) {
    for (int b0 = bl; b0 < bands; b0 += 128) {
      float t[8];
#pragma unroll
      for (int u = 0; u < 8; u++) t[u] = b0 + 16 * u < bands ? part[(int64_t)(b0 + 16 * u) * N + n] : 0.f;
      v += sum8(t);
    }
  }
  red[bl][col] = v;
  __syncthreads();
  if (bl == 0) {
    v = 0.f;
#pragma unroll
    for (int b = 0; b < 16; b++) v += red[b][col];
  }
  return v;
}

// OUT 0: the sum as T;  1: as fp32;  2: the sum is dg, (dh1, dh3) of the SwiGLU as fp32.
template <typename T, int OUT>
__global__ __launch_bounds__(256) void step_bands_kernel(const float* __restrict__ part, int bands, int N, T* __restrict__ y,
                                                         float* __restrict__ f0, float* __restrict__ f1, const T* __restrict__ h1,
                                                         const T* __restrict__ h3) {
  __shared__ float red[16][16];
  const int n = blockIdx.x * 16 + (threadIdx.x & 15);
  const float v = sum_bands16(part, bands, N, n, red);
  if (threadIdx.x >= 16 || n >= N) return;
  if constexpr (OUT == 0) y[n] = from_f32<T>(v);
  else if constexpr (OUT == 1) f0[n] = v;
  else emi_swiglu_adjoint(to_f32(h1[n]), to_f32(h3[n]), v, f0 + n, f1 + n);
}

// Adjoint of y = gamma x rms: from the cotangent of y (the sum of `bands` rows, or T with bands == 0) the one of gamma, and
// the one of x plus the residual's, as fp32 (for the next products) or T.  One block: the vector is short.
template <typename T>
__global__ __launch_bounds__(1024) void step_norm_adjoint_kernel(const float* __restrict__ part, int bands, const T* __restrict__ ct,
                                                                 const T* __restrict__ x, const T* __restrict__ gamma,
                                                                 const float* __restrict__ rms, const float* __restrict__ residual,
                                                                 T* __restrict__ dgamma, float* __restrict__ dx, T* __restrict__ dx_t, int D) {
  extern __shared__ float dy[];                         // [D], then [1024] for band lanes
  __shared__ float scratch[16];
  const float rs = *rms;
  if (bands > 1) {
    // band lanes: as many columns side by side as there are, the threads left share the bands
    const int width = D < 1024 ? D : 1024, lanes = 1024 / width;
    const int bl = threadIdx.x / width, cl = threadIdx.x % width;
    float* red = dy + D;
    for (int n0 = 0; n0 < D; n0 += width) {
      const int n = n0 + cl;
      float v = 0.f;
      if (bl < lanes && n < D) {
        for (int b0 = bl; b0 < bands; b0 += lanes * 8) {
          float t[8];
#pragma unroll
          for (int u = 0; u < 8; u++) t[u] = b0 + lanes * u < bands ? part[(int64_t)(b0 + lanes * u) * D + n] : 0.f;
          v += sum8(t);
        }
      }
      if (lanes > 1) {
        red[threadIdx.x] = v;
        __syncthreads();
        if (bl == 0) {
          v = 0.f;
          for (int l = 0; l < lanes; l++) v += red[l * width + cl];
        }
        __syncthreads();
      }
      if (bl == 0 && n < D) dy[n] = v;
    }
    __syncthreads();
  } else {
    for (int n = threadIdx.x; n < D; n += 1024) dy[n] = bands == 1 ? part[n] : to_f32(ct[n]);
    __syncthreads();
  }
  float dot = 0.f;                                      // sum of dy gamma xhat
  for (int n = threadIdx.x; n < D; n += 1024) dot = fmaf(dy[n] * to_f32(gamma[n]), to_f32(x[n]) * rs, dot);
  const float mean = block_sum_f32(dot, scratch) / D;
  for (int n = threadIdx.x; n < D; n += 1024) {
    const float xh = to_f32(x[n]) * rs, d = dy[n];
    dgamma[n] = from_f32<T>(d * xh);
    float v = rs * (d * to_f32(gamma[n]) - xh * mean);
    if (residual != nullptr) v += residual[n];
    if (dx_t != nullptr) dx_t[n] = from_f32<T>(v);
    else dx[n] = v;
  }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

struct StepDims {
  int64_t L, D, H, heads, pos, table_pairs;
  float eps, scale;
  int dtype;
  int hd() const { return (int)(D / heads); }
  // keys per block: a head in one block while that is a pass of its loads, otherwise enough blocks for the chip
  int kpb() const {
    const int64_t keys = pos + 1;
    if (keys <= 256) return 256;
    const int64_t want = (keys * heads / 512 + 63) / 64 * 64;
    return (int)(want < 128 ? 128 : want > 512 ? 512 : want);
  }
  bool short_cache() const {                              // attention inside the product with wo: step_attention
    const int lanes = hd() / (dtype == EMI_BF16 ? 8 : 4);
    return lanes <= 16 && (heads + 15) / 16 * ((pos + kStepKeys) / kStepKeys) <= kStepRounds;
  }
  int nsplit() const { return (int)((pos + 1 + kpb() - 1) / kpb()); }
};

struct Carve {                                            // consecutive 256-byte aligned pieces of a buffer
  uint8_t* base;
  size_t at = 0;
  template <typename P> P* take(size_t n) {
    P* p = reinterpret_cast<P*>(base + at);
    at += (n * sizeof(P) + 255) / 256 * 256;
    return p;
  }
};

template <typename T> struct Saved {                      // of one layer
  T *x, *q, *k, *v, *att, *x1, *h1, *h3, *g;
  float *lse, *rms1, *rms2;
};
template <typename T> struct SavedAll {
  T* x_out;                                               // the residual stream after the last layer
  float *rms, *part;
};

template <typename T> Saved<T> carve_layer(Carve& c, const StepDims& d) {
  Saved<T> s;
  s.x = c.take<T>(d.D);
  s.q = c.take<T>(d.D);
  s.k = c.take<T>(d.D);
  s.v = c.take<T>(d.D);
  s.att = c.take<T>(d.D);
  s.x1 = c.take<T>(d.D);
  s.h1 = c.take<T>(d.H);
  s.h3 = c.take<T>(d.H);
  s.g = c.take<T>(d.H);
  s.lse = c.take<float>(d.heads);
  s.rms1 = c.take<float>(1);
  s.rms2 = c.take<float>(1);
  return s;
}
template <typename T> SavedAll<T> carve_tail(Carve& c, const StepDims& d) {
  SavedAll<T> s;
  s.x_out = c.take<T>(d.D);
  s.rms = c.take<float>(1);
  s.part = c.take<float>((size_t)d.heads * d.nsplit() * (d.hd() + 2));
  return s;
}
template <typename T> size_t saved_bytes(const StepDims& d) {
  Carve c{nullptr};
  const Saved<T> layer = carve_layer<T>(c, d);
  (void)layer;
  Carve t{nullptr};
  carve_tail<T>(t, d);
  return c.at * (size_t)d.L + t.at;
}

template <typename T>
int step_fwd(hipStream_t st, const void* const* w, const void* x_, const void* kc_, const void* vc_, const float* table, void* y,
             void* saved, const StepDims& d) {
  const T* g1 = (const T*)w[0];
  const T *wq = (const T*)w[1], *wk = (const T*)w[2], *wv = (const T*)w[3], *wo = (const T*)w[4];
  const T* g2 = (const T*)w[5];
  const T *w1 = (const T*)w[6], *w2 = (const T*)w[7], *w3 = (const T*)w[8];
  const T *kc = (const T*)kc_, *vc = (const T*)vc_, *x = (const T*)x_;
  const int64_t D = d.D, H = d.H;
  Carve all{(uint8_t*)saved};
  {
    Carve probe{nullptr};
    carve_layer<T>(probe, d);
    all.at = probe.at * (size_t)d.L;
  }
  SavedAll<T> tail = carve_tail<T>(all, d);
  Carve c{(uint8_t*)saved};
  for (int64_t l = 0; l < d.L; l++) {
    Saved<T> s = carve_layer<T>(c, d);
    T* x_next = tail.x_out;
    if (l + 1 < d.L) {
      Carve ahead = c;
      x_next = carve_layer<T>(ahead, d).x;
    }
    NormGemv<T> a{};
    a.x = x;
    a.gamma = g1 + l * D;
    a.w[0] = wq + l * D * D, a.w[1] = wk + l * D * D, a.w[2] = wv + l * D * D;
    a.y[0] = s.q, a.y[1] = s.k, a.y[2] = s.v;
    a.rms = s.rms1;
    a.table = (const float2*)table;
    a.table_pairs = (int)d.table_pairs;
    a.N = (int)D, a.K = (int)D, a.eps = d.eps;
    if (int rc = launch_norm_gemv<T, 0>(st, a)) return rc;
    if (d.short_cache()) {
      NormGemv<T> o{};
      o.x = x;
      o.w[0] = wo + l * D * D;
      o.y[0] = s.x1;
      o.N = (int)D, o.K = (int)D;
      o.q = s.q, o.k_own = s.k, o.v_own = s.v;
      o.k_cache = kc + l * d.pos * D, o.v_cache = vc + l * d.pos * D;
      o.att = s.att, o.lse = s.lse;
      o.heads = (int)d.heads, o.head_dim = d.hd(), o.keys = (int)d.pos + 1;
      o.scale = d.scale;
      if (int rc = launch_norm_gemv<T, 2>(st, o)) return rc;
    } else {
      if (int rc = launch_llama_step_attn_fwd(st, s.q, kc + l * d.pos * D, vc + l * d.pos * D, s.k, s.v, s.att, s.lse, tail.part,
                                              (int)d.heads, (int)d.pos, d.hd(), d.kpb(), d.scale, d.dtype))
        return rc;
      if (int rc = launch_skinny(st, s.att, wo + l * D * D, x, s.x1, nullptr, 0, 1, D, D, D, D, D, D, 0, 1, d.dtype)) return rc;
    }
    NormGemv<T> f{};
    f.x = s.x1;
    f.gamma = g2 + l * D;
    f.w[0] = w1 + l * H * D, f.w[1] = w3 + l * H * D;
    f.y[0] = s.h1, f.y[1] = s.h3, f.y[2] = s.g;
    f.rms = s.rms2;
    f.N = (int)H, f.K = (int)D, f.eps = d.eps;
    if (int rc = launch_norm_gemv<T, 1>(st, f)) return rc;
    if (int rc = launch_skinny(st, s.g, w2 + l * D * H, s.x1, x_next, nullptr, 0, 1, D, H, H, H, D, D, 0, 1, d.dtype)) return rc;
    x = x_next;
  }
  hipLaunchKernelGGL(step_norm_kernel<T>, dim3(1), dim3(1024), 0, st, x, (const T*)w[9], (T*)y, tail.rms, (int)D, d.eps);
  EMI_CHECK_LAUNCH("emi_llama_step_fwd(norm)");
  return EMI_OK;
}

// Scratch of the reverse pass; L, pos do not enter except through the attention's blocks.
template <typename T> struct BwdWork {
  float *part, *attn, *dx_a, *dx_b, *f0, *f1, *f2, *dsum;
  T *datt, *dk, *dv;
};
template <typename T> BwdWork<T> carve_bwd(Carve& c, const StepDims& d) {
  BwdWork<T> s;
  auto rows = [&](int count, int64_t K, int64_t N) { return (size_t)adjoint_bands<T>(count, (int)K, (int)N) * N; };
  size_t part = rows(1, d.D, d.H);
  for (size_t n : {rows(2, d.H, d.D), rows(1, d.D, d.D), rows(3, d.D, d.D)})
    if (n > part) part = n;
  s.part = c.take<float>(part);
  s.attn = c.take<float>((size_t)d.heads * d.nsplit() * (d.hd() + 2));
  s.dx_a = c.take<float>(d.D);
  s.dx_b = c.take<float>(d.D);
  s.f0 = c.take<float>(d.D > d.H ? d.D : d.H);
  s.f1 = c.take<float>(d.D > d.H ? d.D : d.H);
  s.f2 = c.take<float>(d.D);
  s.dsum = c.take<float>(d.D);
  s.datt = c.take<T>(d.D);
  s.dk = c.take<T>(d.D);
  s.dv = c.take<T>(d.D);
  return s;
}

template <typename T>
int norm_adjoint(hipStream_t st, const BwdWork<T>& k, int bands, const T* ct, const T* x, const T* gamma, const float* rms,
                 const float* residual, T* dgamma, float* dx, T* dx_t, int D) {
  const float* part = k.part;
  if (bands > 1 && (int64_t)bands * D > 96 * 1024) {       // more than one block should sum: its own launch
    hipLaunchKernelGGL((step_bands_kernel<T, 1>), dim3((unsigned)((D + 15) / 16)), dim3(256), 0, st, k.part, bands, D, (T*)nullptr, k.dsum,
                       (float*)nullptr, (const T*)nullptr, (const T*)nullptr);
    EMI_CHECK_LAUNCH("emi_llama_step_bwd(bands)");
    part = k.dsum;
    bands = 1;
  }
  hipLaunchKernelGGL(step_norm_adjoint_kernel<T>, dim3(1), dim3(1024), (size_t)(D + 1024) * sizeof(float), st, part, bands, ct, x, gamma, rms,
                     residual, dgamma, dx, dx_t, D);
  EMI_CHECK_LAUNCH("emi_llama_step_bwd(norm)");
  return EMI_OK;
}

template <typename T>
int step_bwd(hipStream_t st, const void* const* w, const void* x_, const void* kc_, const void* vc_, const float* table, const void* saved,
             const void* dy, void* const* grads, void* workspace, const StepDims& d) {
  const T* g1 = (const T*)w[0];
  const T *wq = (const T*)w[1], *wk = (const T*)w[2], *wv = (const T*)w[3], *wo = (const T*)w[4];
  const T* g2 = (const T*)w[5];
  const T *w1 = (const T*)w[6], *w2 = (const T*)w[7], *w3 = (const T*)w[8];
  const T *kc = (const T*)kc_, *vc = (const T*)vc_;
  T* const* gr = (T* const*)grads;      // dx, then the ten weights in the order of w, then the caches
  const int64_t D = d.D, H = d.H;
  Carve wsc{(uint8_t*)workspace};
  BwdWork<T> k = carve_bwd<T>(wsc, d);
  Carve probe{nullptr};
  carve_layer<T>(probe, d);
  const size_t layer_bytes = probe.at;
  Carve all{(uint8_t*)const_cast<void*>(saved), layer_bytes * (size_t)d.L};
  SavedAll<T> tail = carve_tail<T>(all, d);
  float *dx = k.dx_a, *dx1 = k.dx_b;
  if (int rc = norm_adjoint<T>(st, k, 0, (const T*)dy, tail.x_out, (const T*)w[9], tail.rms, nullptr, gr[10], dx, nullptr, (int)D)) return rc;
  for (int64_t l = d.L - 1; l >= 0; l--) {
    Carve c{(uint8_t*)const_cast<void*>(saved), layer_bytes * (size_t)l};
    const Saved<T> s = carve_layer<T>(c, d);
    const T* x = l == 0 ? (const T*)x_ : s.x;
    int bands = 1;
    Adjoint<T> a{};
    a.w[0] = w2 + l * D * H, a.dw[0] = gr[8] + l * D * H, a.dy[0] = dx;                       // w2 [D, H]
    a.x = s.g, a.part = k.part, a.count = 1, a.K = (int)D, a.N = (int)H;
    if (int rc = launch_adjoint<T>(st, a, &bands)) return rc;
    hipLaunchKernelGGL((step_bands_kernel<T, 2>), dim3((unsigned)((H + 15) / 16)), dim3(256), 0, st, k.part, bands, (int)H, (T*)nullptr, k.f0,
                       k.f1, s.h1, s.h3);
    EMI_CHECK_LAUNCH("emi_llama_step_bwd(swiglu)");
    a = Adjoint<T>{};
    a.w[0] = w1 + l * H * D, a.dw[0] = gr[7] + l * H * D, a.dy[0] = k.f0;                     // w1, w3 [H, D]
    a.w[1] = w3 + l * H * D, a.dw[1] = gr[9] + l * H * D, a.dy[1] = k.f1;
    a.x = s.x1, a.gamma = g2 + l * D, a.rms = s.rms2, a.part = k.part, a.count = 2, a.K = (int)H, a.N = (int)D;
    if (int rc = launch_adjoint<T>(st, a, &bands)) return rc;
    if (int rc = norm_adjoint<T>(st, k, bands, nullptr, s.x1, g2 + l * D, s.rms2, dx, gr[6] + l * D, dx1, nullptr, (int)D)) return rc;
    a = Adjoint<T>{};
    a.w[0] = wo + l * D * D, a.dw[0] = gr[5] + l * D * D, a.dy[0] = dx1;                      // wo [D, D]
    a.x = s.att, a.part = k.part, a.count = 1, a.K = (int)D, a.N = (int)D;
    if (int rc = launch_adjoint<T>(st, a, &bands)) return rc;
    hipLaunchKernelGGL((step_bands_kernel<T, 0>), dim3((unsigned)((D + 15) / 16)), dim3(256), 0, st, k.part, bands, (int)D, k.datt,
                       (float*)nullptr, (float*)nullptr, (const T*)nullptr, (const T*)nullptr);
    EMI_CHECK_LAUNCH("emi_llama_step_bwd(sum)");
    const int64_t cache = l * d.pos * D;
    if (int rc = launch_llama_step_attn_bwd(st, s.q, kc + cache, vc + cache, s.k, s.v, s.att, s.lse, k.datt, gr[11] + cache, gr[12] + cache,
                                            k.dk, k.dv, k.attn, table, (int)d.table_pairs, k.f0, k.f1, k.f2, (int)d.heads, (int)d.pos, d.hd(),
                                            d.kpb(), d.scale, d.dtype))
      return rc;
    a = Adjoint<T>{};
    a.w[0] = wq + l * D * D, a.dw[0] = gr[2] + l * D * D, a.dy[0] = k.f0;
    a.w[1] = wk + l * D * D, a.dw[1] = gr[3] + l * D * D, a.dy[1] = k.f1;
    a.w[2] = wv + l * D * D, a.dw[2] = gr[4] + l * D * D, a.dy[2] = k.f2;
    a.x = x, a.gamma = g1 + l * D, a.rms = s.rms1, a.part = k.part, a.count = 3, a.K = (int)D, a.N = (int)D;
    if (int rc = launch_adjoint<T>(st, a, &bands)) return rc;
    if (int rc = norm_adjoint<T>(st, k, bands, nullptr, x, g1 + l * D, s.rms1, dx1, gr[1] + l * D, dx, l == 0 ? gr[0] : nullptr, (int)D))
      return rc;
  }
  return EMI_OK;
}

bool dims_ok(const StepDims& d) {
  const int64_t V = d.dtype == EMI_BF16 ? 8 : 4;
  // LDS: the padded vector of the product kernel, the vector of the norm's adjoint
  return (d.dtype == EMI_BF16 || d.dtype == EMI_F32) && d.L > 0 && d.D > 0 && d.H > 0 && d.heads > 0 && d.D % d.heads == 0 &&
         d.D % V == 0 && d.H % V == 0 && d.hd() % V == 0 && d.hd() <= 256 && d.D <= 8192 && d.H <= (1 << 20) && d.heads <= 65535 && d.pos > 0 &&
         d.pos < (1 << 30) && d.table_pairs > 0 && (d.D / 2) % d.table_pairs == 0;
}

}  // namespace
}  // namespace emi

using namespace emi;

extern "C" size_t emi_llama_step_saved_bytes(int64_t layers, int64_t dim, int64_t hidden, int64_t heads, int64_t pos, int dtype) {
  const StepDims d{layers, dim, hidden, heads, pos, 1, 0.f, 0.f, dtype};
  if (!dims_ok(d)) return 0;
  return dtype == EMI_BF16 ? saved_bytes<bf16>(d) : saved_bytes<float>(d);
}

extern "C" size_t emi_llama_step_bwd_workspace_bytes(int64_t layers, int64_t dim, int64_t hidden, int64_t heads, int64_t pos, int dtype) {
  const StepDims d{layers, dim, hidden, heads, pos, 1, 0.f, 0.f, dtype};
  if (!dims_ok(d)) return 0;
  Carve c{nullptr};
  if (dtype == EMI_BF16) carve_bwd<bf16>(c, d);
  else carve_bwd<float>(c, d);
  return c.at;
}

static int check_step_call(const char* name, const StepDims& d, const void* const* weights, std::initializer_list<const void*> ptrs) {
  EMI_REQUIRE(dims_ok(d), "%s: unsupported shape (layers=%lld dim=%lld hidden=%lld heads=%lld pos=%lld dtype=%d)", name, (long long)d.L,
              (long long)d.D, (long long)d.H, (long long)d.heads, (long long)d.pos, d.dtype);
  EMI_REQUIRE(weights != nullptr, "%s: null weight table", name);
  for (int i = 0; i < 10; i++)
    EMI_REQUIRE(weights[i] != nullptr && (reinterpret_cast<uintptr_t>(weights[i]) & 15) == 0, "%s: weight %d is null or not 16-byte aligned", name, i);
  for (const void* p : ptrs)
    EMI_REQUIRE(p != nullptr && (reinterpret_cast<uintptr_t>(p) & 15) == 0, "%s: a buffer is null or not 16-byte aligned", name);
  return EMI_OK;
}

extern "C" int emi_llama_step_fwd(emi_stream_t stream, const void* const* weights, const void* x, const void* key_cache,
                                  const void* value_cache, const float* rope_table, int64_t table_pairs, void* y, void* saved,
                                  size_t saved_bytes_given, int64_t layers, int64_t dim, int64_t hidden, int64_t heads, int64_t pos,
                                  float eps, float scale, int dtype) {
  const StepDims d{layers, dim, hidden, heads, pos, table_pairs, eps, scale, dtype};
  if (int rc = check_step_call("emi_llama_step_fwd", d, weights, {x, key_cache, value_cache, rope_table, y, saved})) return rc;
  const size_t need = emi_llama_step_saved_bytes(layers, dim, hidden, heads, pos, dtype);
  EMI_REQUIRE(saved_bytes_given >= need, "emi_llama_step_fwd: %zu bytes of saved values needed, got %zu", need, saved_bytes_given);
  hipStream_t st = static_cast<hipStream_t>(stream);
  return dtype == EMI_BF16 ? step_fwd<bf16>(st, weights, x, key_cache, value_cache, rope_table, y, saved, d)
                           : step_fwd<float>(st, weights, x, key_cache, value_cache, rope_table, y, saved, d);
}

extern "C" int emi_llama_step_bwd(emi_stream_t stream, const void* const* weights, const void* x, const void* key_cache,
                                  const void* value_cache, const float* rope_table, int64_t table_pairs, const void* saved, const void* dy,
                                  void* const* grads, void* workspace, size_t workspace_bytes, int64_t layers, int64_t dim, int64_t hidden,
                                  int64_t heads, int64_t pos, float eps, float scale, int dtype) {
  const StepDims d{layers, dim, hidden, heads, pos, table_pairs, eps, scale, dtype};
  if (int rc = check_step_call("emi_llama_step_bwd", d, weights, {x, key_cache, value_cache, rope_table, saved, dy, workspace})) return rc;
  EMI_REQUIRE(grads != nullptr, "emi_llama_step_bwd: null gradient table");
  for (int i = 0; i < 13; i++)
    EMI_REQUIRE(grads[i] != nullptr && (reinterpret_cast<uintptr_t>(grads[i]) & 15) == 0,
                "emi_llama_step_bwd: gradient %d is null or not 16-byte aligned", i);
  const size_t need = emi_llama_step_bwd_workspace_bytes(layers, dim, hidden, heads, pos, dtype);
  EMI_REQUIRE(workspace_bytes >= need, "emi_llama_step_bwd: workspace of %zu bytes needed, got %zu", need, workspace_bytes);
  hipStream_t st = static_cast<hipStream_t>(stream);
  return dtype == EMI_BF16 ? step_bwd<bf16>(st, weights, x, key_cache, value_cache, rope_table, saved, dy, grads, workspace, d)
                           : step_bwd<float>(st, weights, x, key_cache, value_cache, rope_table, saved, dy, grads, workspace, d);
}
