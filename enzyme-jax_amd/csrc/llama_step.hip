// The reference's own program as one call each way: a decoder step of one token through all layers (test/llama.py:35-238)
// and its reverse (every weight and both caches).
//
// Small models are a chain of launches, each as long as its latencies (a few us), and large ones are bound by the weights,
// which are read once (and, in reverse, read and written once).  Both want the fewest kernels: what lies between two
// matrix-vector products - RMSNorm, the rotation, SwiGLU, residuals, the new cache row - is done where its operand is
// loaded or its result leaves, and the cache is not copied to append a row to it.
//   forward, per layer:  norm + wq,wk,wv + rotation | attention over cache and own row (| combine) | wo + residual |
//                        norm + w1,w3 + SwiGLU | w2 + residual;  with a short cache attention + wo + residual are one, with a longer
//                        one combine + wo + residual
//   reverse, per layer:  norm' + w2^T dy and dw2 | SwiGLU' + w1^T dh1 + w3^T dh3 and dw1, dw3 | norm' + wo^T dy and dwo |
//                        attention' | inverse rotation + wq^T dq + ... and dwq, dwk, dwv
// The forward call leaves what the reverse one needs in `saved`.
// Measured against the same step operator by operator (us): dim 288, 6 layers, fp32: forward 1071 -> 100 (99 launches ->
// 25), with the reverse from StableHLO text at position 255 4042 -> 315 (289 launches -> 63); dim 4096, 2 layers, bf16,
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
                               const void* v_tail, const void* o, const float* lse, const float* do_part, int do_bands, void* dk_cache,
                               void* dv_cache, void* dk_tail, void* dv_tail, float* part, int heads, int pos, int head_dim, int keys_per_block,
                               float scale, int dtype);

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
// MODE 1, row p of w0 and of w1 (h1, h3 of the SwiGLU); MODE 2 and 3, rows 2p and 2p + 1 of w0 (wo) times the attention's result,
// which each block works out for itself, from the keys and values (2: step_attention) or by adding up its key blocks' shares (3:
// step_combine).  The rows stream through in batches of UN 16-byte pieces per lane,
// the next pair's first batch requested while the current one is summed, and the first pair's before the block normalises
// the vector: each block keeps gamma x / rms(x) in LDS (the two halves of an eight-element piece apart, so that a
// lane's reads of 16 bytes do not collide).
template <typename T> struct NormGemv {
  const T *x, *gamma;    // MODE 2, 3: x is the residual
  const T* w[3];
  T* y[3];               // MODE 0: q, k, v;  MODE 1: h1, h3, g;  MODE 2, 3: x + w0 att
  float* rms;            // 1 / rms(x), for the adjoint
  const float2* table;   // MODE 0: (cos, sin) of pair i at i % table_pairs
  int N, K, table_pairs;
  float eps;
  // MODE 2: the attention whose result the vector is;  MODE 3: its shares [heads][shares][head_dim + 2] (sum, maximum, weight)
  const float* part;
  int shares;
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

// att of one query from its key blocks' shares, into the vector's LDS image: a 16-byte piece a thread, eight shares requested
// together.  One such round is a latency of the L2 where a launch that adds the shares up is 3 to 5 us; and with the launch gone
// a short cache is dealt to more blocks.  Where
// StepDims::combines() says so.  Forward replayed, us, a launch | this (shares, rounds): 4 layers at dim 512 fp32, 255 keys 87.3 | 80.6 (4, 1), 700
// 92.4 | 87.3 (11, 2), 2000 97.5 | 91.8 (16, 2); dim 1024 bf16, 2000 keys 115 | 108; 2 layers at dim 2048 fp32, 255 keys 149 | 116 (4, 2), at 4096 338 | 314
// (4, 4).  More: dim 768 fp32, 2000 keys 116 | 122 (32, 4), dim 2048 bf16 99 | 105 (32, 4), dim 4096 bf16, 4095 keys 205 | 210 (16, 4).
constexpr int kCombineShares = 8;
template <typename T> __device__ __forceinline__ void step_combine(const NormGemv<T>& a, float* xs, int pieces, bool store) {
  constexpr int V = ChunkCached<T>::N;
  const int stride = a.head_dim + 2;
  for (int c = threadIdx.x; c * V < a.K; c += 256) {
    const int h = c * V / a.head_dim, e0 = c * V - h * a.head_dim;
    const float* p0 = a.part + (int64_t)h * a.shares * stride;
    float acc[V], mx = -INFINITY, sum = 0.f;
#pragma unroll
    for (int e = 0; e < V; e++) acc[e] = 0.f;
    for (int s0 = 0; s0 < a.shares; s0 += kCombineShares) {
      float2 v[kCombineShares][V / 2], st[kCombineShares];
#pragma unroll
      for (int u = 0; u < kCombineShares; u++) {           // past the last: it again, of weight zero
        const float* p = p0 + (s0 + u < a.shares ? s0 + u : a.shares - 1) * stride;
        st[u] = *reinterpret_cast<const float2*>(p + a.head_dim);
#pragma unroll
        for (int e = 0; e < V / 2; e++) v[u][e] = *reinterpret_cast<const float2*>(p + e0 + 2 * e);
      }
      float nm = mx;
#pragma unroll
      for (int u = 0; u < kCombineShares; u++) nm = fmaxf(nm, st[u].x);
      const float alpha = mx == -INFINITY ? 0.f : __expf(mx - nm);
      sum *= alpha;
#pragma unroll
      for (int e = 0; e < V; e++) acc[e] *= alpha;
      mx = nm;
#pragma unroll
      for (int u = 0; u < kCombineShares; u++) {
        if (s0 + u >= a.shares) continue;
        const float w = st[u].x == -INFINITY ? 0.f : __expf(st[u].x - mx);      // (times a NaN it stays one)
        sum = fmaf(w, st[u].y, sum);
#pragma unroll
        for (int e = 0; e < V / 2; e++) {
          acc[2 * e] = fmaf(w, v[u][e].x, acc[2 * e]);
          acc[2 * e + 1] = fmaf(w, v[u][e].y, acc[2 * e + 1]);
        }
      }
    }
    const float inv = 1.0f / sum;
#pragma unroll
    for (int e = 0; e < V; e++) acc[e] = round_to<T>(acc[e] * inv);
    if (store) {
      ChunkCached<T>::store(a.att + c * V, acc);
      if (e0 == 0) a.lse[h] = mx + __logf(sum);
    }
#pragma unroll
    for (int g = 0; g < V / 4; g++)
      *reinterpret_cast<f4*>(xs + (g * pieces + c) * 4) = f4{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
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
    if constexpr (MODE >= 2) {
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
  if constexpr (MODE >= 2) {
    if constexpr (MODE == 2) step_attention<T>(a, xs, pieces, blockIdx.x == 0);
    else step_combine<T>(a, xs, pieces, blockIdx.x == 0);
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
    if constexpr (MODE >= 2) {                             // rows and residual in fp32, rounded once
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
// Every row of a matrix is read once (for the cotangent of x) while its gradient's row is written; HBM-bound on both.  A block
// owns `width` 16-byte pieces of columns and a band of rows; its row lanes (256 / width) take the band's rows in turn, two
// register sets of UN rows in flight, and meet in the wavefront and through LDS.  The bands' sums [bands][N] go to `part` in fp32.
//
// What lies between two such products needs a value of every band: the norm's adjoint, the SwiGLU's, the inverse rotation.  The
// kernel behind works it out itself, for its band's rows alone, while its first rows of W are on their way, so bands are few
// (kMostBands of narrow blocks; more only so that a band has at most kMostRows rows) and the norm's one sum over all columns, which is linear in them, arrives as a share
// of every block (`dots`).  Five launches a layer; nine when the bands were 96 and their sums launches of their own (a
// norm's 5.7 us of one block, the others 2.6).
template <typename T> struct Adjoint {
  const T* w[3];
  T* dw[3];
  const T *x, *gamma;      // the products' operand: x, or with gamma the normalised gamma x rms
  const float* rms;
  float *part, *dots;      // results; dots, with gamma: each block's share of the sum over the columns of part gamma x rms
  int count, K, N, rows_per_band, width;
  // the rows' cotangent: from the sums of the product behind, [in_bands][K]
  const float *in, *in_dots;
  int in_bands, in_ndots;
  const T *nx, *ngamma;    // kNorm: the norm between, of nx; its adjoint plus `residual` leaves as dx (fp32) or dx_t
  const float *nrms, *residual;
  float* dx;
  T *dx_t, *dgamma;
  const T *h1, *h3;        // kSwiglu
  const T *dk, *dv;        // kAttention: in is [heads][in_bands][head_dim + 2], dq's shares; dk, dv of the token's own row
  const float2* table;
  int table_pairs, head_dim;
};
enum { kNorm, kSwiglu, kAttention };

// In pairs: added one by one the bands' sums decided the error.
template <int N> __device__ __forceinline__ float sum_pairs(float (&t)[N]) {
#pragma unroll
  for (int n = N / 2; n > 0; n /= 2)
#pragma unroll
    for (int i = 0; i < n; i++) t[i] += t[i + n];
  return t[0];
}
// The sum of n values `stride` apart, by four neighbouring lanes; all four receive it.  Unconditional loads: the compiler
// waits for each guarded one.
__device__ __forceinline__ float bands_sum(const float* __restrict__ p, int64_t stride, int n) {
  float v = 0.f;
  for (int b0 = threadIdx.x & 3; b0 < n; b0 += 32) {
    float t[8];
#pragma unroll
    for (int u = 0; u < 8; u++) t[u] = p[(b0 + 4 * u < n ? b0 + 4 * u : b0) * stride];
#pragma unroll
    for (int u = 0; u < 8; u++) t[u] = b0 + 4 * u < n ? t[u] : 0.f;
    v += sum_pairs(t);
  }
  return quad_sum(v);
}

// The cotangent of rows r_begin .. r_end, into LDS; four lanes a row.  The norm's mean needs the whole block: the first rows' sums
// are requested before it.
template <typename T, int FROM>
__device__ __forceinline__ void rows_cotangent(const Adjoint<T>& a, int r_begin, int r_end, bool write, float* dy, float* scratch) {
  const bool first = (threadIdx.x & 3) == 0;
  int r = r_begin + (threadIdx.x >> 2);
  if constexpr (FROM == kNorm) {
    float dot = 0.f;
    for (int i = threadIdx.x; i < a.in_ndots; i += 256) dot += a.in_dots[i];
    const float rs = *a.nrms;
    float d = 0.f, g = 0.f, xh = 0.f, res = 0.f;
    auto load = [&]() {
      if (r < r_end) {
        g = to_f32(a.ngamma[r]);
        xh = to_f32(a.nx[r]) * rs;
        if (a.residual != nullptr) res = a.residual[r];
        d = bands_sum(a.in + r, a.K, a.in_bands);
      }
    };
    load();
    const float mean = block_sum_f32(dot, scratch) / a.K;
    while (r < r_end) {
      const float o = rs * (d * g - xh * mean) + res;
      if (write && first) {
        a.dgamma[r] = from_f32<T>(d * xh);
        if (a.dx_t != nullptr) a.dx_t[r] = from_f32<T>(o);
        else a.dx[r] = o;
      }
      if (first) dy[r - r_begin] = o;
      r += 64;
      load();
    }
    return;
  }
  for (; r < r_end; r += 64) {
    float o;
    if constexpr (FROM == kSwiglu) {
      const int k = r < a.K ? r : r - a.K;
      float d1, d3;
      emi_swiglu_adjoint(to_f32(a.h1[k]), to_f32(a.h3[k]), bands_sum(a.in + k, a.K, a.in_bands), &d1, &d3);
      o = r < a.K ? d1 : d3;
    } else {                                               // the rows of a pair turned back by the position's angle
      const int m = r / a.K, k = r - m * a.K;
      if (m == 2) {
        o = to_f32(a.dv[k]);
      } else {
        const int h = k / a.head_dim, e = k - h * a.head_dim;
        float own, other;
        if (m == 0) {
          const float* p = a.in + (int64_t)h * a.in_bands * (a.head_dim + 2);
          own = bands_sum(p + e, a.head_dim + 2, a.in_bands);
          other = bands_sum(p + (e ^ 1), a.head_dim + 2, a.in_bands);
        } else {
          own = to_f32(a.dk[k]);
          other = to_f32(a.dk[k ^ 1]);
        }
        const float2 t = a.table[(k >> 1) % a.table_pairs];
        o = (k & 1) == 0 ? t.x * own + t.y * other : t.x * own - t.y * other;
      }
    }
    if (first) dy[r - r_begin] = o;
  }
}

template <typename T, int FROM, bool STREAM>
__global__ __launch_bounds__(256) void step_adjoint_kernel(Adjoint<T> a) {
  using Raw = typename ChunkCached<T>::Raw;
  constexpr int V = ChunkCached<T>::N, UN = 8;
  extern __shared__ float dy[];                            // [rows_per_band]
  __shared__ float red[4][64][V + 1];
  __shared__ float scratch[4];
  const int pieces = a.N / V, lanes = 256 / a.width;
  const int rl = threadIdx.x / a.width, cl = threadIdx.x % a.width;
  const int piece = blockIdx.x * a.width + cl, n = piece * V;
  const bool live = piece < pieces;
  const int total = a.count * a.K;
  const int r_begin = blockIdx.y * a.rows_per_band, r_end = r_begin + a.rows_per_band < total ? r_begin + a.rows_per_band : total;
  float acc[V], xv[V], gx[V];                              // gx: gamma x rms before it is rounded
#pragma unroll
  for (int e = 0; e < V; e++) acc[e] = xv[e] = gx[e] = 0.f;
  auto matrix = [&](int r) { return a.count == 1 ? 0 : r / a.K; };
  auto pick = [](auto&& p, int m) { return m == 0 ? p[0] : m == 1 ? p[1] : p[2]; };
  auto issue = [&](int r0, Raw(&w)[UN]) {
#pragma unroll
    for (int u = 0; u < UN; u++) {
      const int r = r0 + u * lanes < r_end ? r0 + u * lanes : r_end - 1;            // past the band: its last row, unused
      const int m = matrix(r), k = r - m * a.K;
      w[u] = Chunk<T>::load_raw(pick(a.w, m) + (int64_t)k * a.N + n);
    }
  };
  auto consume = [&](int r0, const Raw(&w)[UN]) {
#pragma unroll
    for (int u = 0; u < UN; u++) {
      const int r = r0 + u * lanes;
      if (r < r_end) {
        const int m = matrix(r), k = r - m * a.K;
        const float d = dy[r - r_begin];
        float wv[V], o[V];
        ChunkCached<T>::unpack(w[u], wv);
#pragma unroll
        for (int e = 0; e < V; e++) {
          acc[e] = fmaf(d, wv[e], acc[e]);
          o[e] = d * xv[e];
        }
        T* dst = pick(a.dw, m) + (int64_t)k * a.N + n;
        if constexpr (STREAM) Chunk<T>::store(dst, o);
        else ChunkCached<T>::store(dst, o);
      }
    }
  };
  Raw w0[UN], w1[UN];
  int r = r_begin + rl;
  if (live) {
    if (r < r_end) issue(r, w0);
    ChunkCached<T>::load(a.x + n, xv);
    if (a.gamma != nullptr) {
      float gv[V];
      ChunkCached<T>::load(a.gamma + n, gv);
      const float rs = *a.rms;
#pragma unroll
      for (int e = 0; e < V; e++) {
        gx[e] = gv[e] * (xv[e] * rs);
        xv[e] = round_to<T>(gx[e]);
      }
    }
  }
  rows_cotangent<T, FROM>(a, r_begin, r_end, blockIdx.x == 0, dy, scratch);
  __syncthreads();
  if (live) {
    while (r < r_end) {
      const int r1 = r + UN * lanes;
      if (r1 < r_end) issue(r1, w1);
      consume(r, w0);
      if (r1 >= r_end) break;
      r = r1 + UN * lanes;
      if (r < r_end) issue(r, w0);
      consume(r1, w1);
    }
  }
  // the row lanes of a wavefront, then the wavefronts
#pragma unroll
  for (int e = 0; e < V; e++) {
    if (a.width <= 32) acc[e] = sum_xor32(acc[e]);
    if (a.width <= 16) acc[e] = sum_xor16(acc[e]);
    if (a.width <= 8) acc[e] += ror16<8>(acc[e]);
    red[threadIdx.x >> 6][threadIdx.x & 63][e] = acc[e];
  }
  __syncthreads();
  if (threadIdx.x >= 64) return;
  float dot = 0.f;
  if ((int)threadIdx.x < a.width && live) {
#pragma unroll
    for (int e = 0; e < V; e++) {
      acc[e] = (red[0][threadIdx.x][e] + red[1][threadIdx.x][e]) + (red[2][threadIdx.x][e] + red[3][threadIdx.x][e]);
      dot = fmaf(acc[e], gx[e], dot);
    }
    float* dst = a.part + (int64_t)blockIdx.y * a.N + n;
#pragma unroll
    for (int e = 0; e < V; e += 4) *reinterpret_cast<f4*>(dst + e) = f4{acc[e], acc[e + 1], acc[e + 2], acc[e + 3]};
  }
  if (a.gamma == nullptr) return;
  dot = wave_sum(dot);
  if (threadIdx.x == 0) a.dots[blockIdx.y * gridDim.x + blockIdx.x] = dot;
}

// Blocks: as narrow as leaves eight of them side by side (a row's share is at least 128 bytes), so that bands are few, and about
// two per CU where there are rows enough, at least two a row lane.
constexpr int kMostBands = 64, kMostRows = 4096;           // rows: of a band, their cotangent stands in LDS
struct AdjointGrid { int width, cols, bands, rows_per_band; };
template <typename T> AdjointGrid adjoint_grid(int count, int K, int N) {
  constexpr int V = ChunkCached<T>::N;
  const int pieces = N / V, total = count * K;
  AdjointGrid g;
  g.width = 64;
  while (g.width > 8 && pieces < 8 * g.width) g.width /= 2;
  g.cols = (pieces + g.width - 1) / g.width;
  const int lanes = 256 / g.width, most = (total + 2 * lanes - 1) / (2 * lanes);
  int bands = (512 + g.cols - 1) / g.cols;
  if (bands > most) bands = most;
  if (bands > kMostBands) bands = kMostBands;
  if (bands < (total + kMostRows - 1) / kMostRows) bands = (total + kMostRows - 1) / kMostRows;
  g.rows_per_band = (total + bands - 1) / bands;
  g.bands = (total + g.rows_per_band - 1) / g.rows_per_band;
  return g;
}

template <typename T, int FROM> int launch_adjoint(hipStream_t st, Adjoint<T> a, const AdjointGrid& g) {
  a.width = g.width;
  a.rows_per_band = g.rows_per_band;
  const dim3 grid((unsigned)g.cols, (unsigned)g.bands);
  const size_t lds = (size_t)g.rows_per_band * sizeof(float);
  if ((size_t)a.count * a.K * a.N * sizeof(T) > ((size_t)32 << 20))
    hipLaunchKernelGGL((step_adjoint_kernel<T, FROM, true>), grid, dim3(256), lds, st, a);
  else
    hipLaunchKernelGGL((step_adjoint_kernel<T, FROM, false>), grid, dim3(256), lds, st, a);
  EMI_CHECK_LAUNCH("emi_llama_step(adjoint products)");
  return EMI_OK;
}

// The first norm's adjoint of the reverse pass, whose cotangent is the caller's: one band and its dot.  One block: the vector is short.
template <typename T>
__global__ __launch_bounds__(1024) void step_cotangent_kernel(const T* __restrict__ ct, const T* __restrict__ x, const T* __restrict__ gamma,
                                                              const float* __restrict__ rms, float* __restrict__ part, float* __restrict__ dots,
                                                              int D) {
  __shared__ float scratch[16];
  const float rs = *rms;
  float dot = 0.f;
  for (int n = threadIdx.x; n < D; n += 1024) {
    const float d = to_f32(ct[n]);
    part[n] = d;
    dot = fmaf(d, to_f32(gamma[n]) * (to_f32(x[n]) * rs), dot);
  }
  dot = block_sum_f32(dot, scratch);
  if (threadIdx.x == 0) *dots = dot;
}
// The last one's, which no product follows: 64 columns a block.
template <typename T> __global__ __launch_bounds__(256) void step_norm_rows_kernel(Adjoint<T> a) {
  __shared__ float dy[64], scratch[4];
  const int r0 = blockIdx.x * 64;
  rows_cotangent<T, kNorm>(a, r0, r0 + 64 < a.K ? r0 + 64 : a.K, true, dy, scratch);
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

struct StepDims {
  int64_t L, D, H, heads, pos, table_pairs;
  float eps, scale;
  int dtype;
  int hd() const { return (int)(D / heads); }
  // keys per block: enough blocks for the chip; as few as 64 where the product behind adds up their shares and that costs less than
  // one block's longer chain of keys, otherwise a head in one block while that is a pass of its loads.  From 224 keys, and with two
  // pieces of a head a lane, whose chain is six times as long a key, from 96.  us, one block | 64 keys: dim 1024 fp32, 4 layers, 72
  // keys 111 | 116, 151 keys 115 | 117, 256 keys 120 | 117; dim 2048 bf16, 72 keys 88 | 91; in two pieces, dim 4096 fp32, 2 layers,
  // 72 keys 300 | 305, 121 keys 311 | 305
  int kpb() const {
    const int64_t keys = pos + 1, want = (keys * heads / 512 + 63) / 64 * 64;
    const int64_t fine = want < 64 ? 64 : want > 512 ? 512 : want;
    const int64_t from = hd() / (dtype == EMI_BF16 ? 8 : 4) > 16 ? 96 : 224;
    if (keys >= from && combines((keys + fine - 1) / fine)) return (int)fine;
    if (keys <= 256) return 256;
    return (int)(want < 128 ? 128 : want > 512 ? 512 : want);
  }
  // step_combine's rounds of loads, and whether the product with wo adds up this many shares a head: two rounds, or more of at most
  // eight shares
  int64_t rounds(int64_t shares) const { return (D / (dtype == EMI_BF16 ? 8 : 4) + 255) / 256 * ((shares + kCombineShares - 1) / kCombineShares); }
  bool combines(int64_t shares) const { return rounds(shares) <= 2 || (shares <= kCombineShares && rounds(shares) <= 4); }
  // (four rounds only with the blocks of 64 keys that they allow: dim 4096 fp32, 2 layers, us, a launch | inside, 300 keys in blocks of 64
  // 315 | 308, 512 to 1023 keys in blocks of 128 317 to 319 | 320 to 322)
  bool combine_inside() const { return nsplit() > 1 && combines(nsplit()) && (rounds(nsplit()) <= 2 || kpb() == 64); }
  bool short_cache() const {                              // attention inside the product with wo: step_attention
    const int lanes = hd() / (dtype == EMI_BF16 ? 8 : 4);
    return lanes <= 16 && (heads + 15) / 16 * ((pos + kStepKeys) / kStepKeys) <= kStepRounds;
  }
  int nsplit() const { return (int)((pos + 1 + kpb() - 1) / kpb()); }
  // the adjoint's: the product behind adds up its blocks' shares, so 64 keys, one pass of its loads, until they fill the chip
  int kpb_bwd() const {
    const int64_t want = ((pos + 1) * heads / 512 + 63) / 64 * 64;
    return (int)(want < 64 ? 64 : want > 512 ? 512 : want);
  }
  int nsplit_bwd() const { return (int)((pos + kpb_bwd()) / kpb_bwd()); }
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
      const bool inside = d.combine_inside();
      if (int rc = launch_llama_step_attn_fwd(st, s.q, kc + l * d.pos * D, vc + l * d.pos * D, s.k, s.v, inside ? nullptr : s.att, s.lse, tail.part,
                                              (int)d.heads, (int)d.pos, d.hd(), d.kpb(), d.scale, d.dtype))
        return rc;
      if (inside) {
        NormGemv<T> o{};
        o.x = x;
        o.w[0] = wo + l * D * D;
        o.y[0] = s.x1;
        o.N = (int)D, o.K = (int)D;
        o.part = tail.part, o.shares = d.nsplit();
        o.att = s.att, o.lse = s.lse;
        o.heads = (int)d.heads, o.head_dim = d.hd();
        if (int rc = launch_norm_gemv<T, 3>(st, o)) return rc;
      } else if (int rc = launch_skinny(st, s.att, wo + l * D * D, x, s.x1, nullptr, 0, 1, D, D, D, D, D, D, 0, 1, d.dtype)) return rc;
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

// Scratch of the reverse pass; L does not enter, pos only through the attention's blocks.  A product reads the sums of the one
// before while it leaves its own: two sets.
template <typename T> struct BwdWork {
  float *part[2], *dots, *attn, *dx_a, *dx_b;
  T *dk, *dv;
};
template <typename T> BwdWork<T> carve_bwd(Carve& c, const StepDims& d) {
  BwdWork<T> s;
  size_t part = (size_t)d.D, dots = 1;
  auto take = [&](int count, int64_t K, int64_t N) {
    const AdjointGrid g = adjoint_grid<T>(count, (int)K, (int)N);
    if ((size_t)g.bands * N > part) part = (size_t)g.bands * N;
    if ((size_t)g.bands * g.cols > dots) dots = (size_t)g.bands * g.cols;
  };
  take(1, d.D, d.H);
  take(2, d.H, d.D);
  take(1, d.D, d.D);
  take(3, d.D, d.D);
  for (float*& p : s.part) p = c.take<float>(part);
  s.dots = c.take<float>(dots);
  s.attn = c.take<float>((size_t)d.heads * d.nsplit_bwd() * (d.hd() + 2));
  s.dx_a = c.take<float>(d.D);
  s.dx_b = c.take<float>(d.D);
  s.dk = c.take<T>(d.D);
  s.dv = c.take<T>(d.D);
  return s;
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
  const AdjointGrid gw2 = adjoint_grid<T>(1, (int)D, (int)H), gw13 = adjoint_grid<T>(2, (int)H, (int)D), gwo = adjoint_grid<T>(1, (int)D, (int)D),
                    gqkv = adjoint_grid<T>(3, (int)D, (int)D);
  hipLaunchKernelGGL(step_cotangent_kernel<T>, dim3(1), dim3(1024), 0, st, (const T*)dy, tail.x_out, (const T*)w[9], tail.rms, k.part[1], k.dots,
                     (int)D);
  EMI_CHECK_LAUNCH("emi_llama_step_bwd(cotangent)");
  // what the norm between two products needs: of the layer's input, or of the result
  Adjoint<T> norm{};
  norm.in = k.part[1], norm.in_dots = k.dots, norm.in_bands = norm.in_ndots = 1;
  norm.nx = tail.x_out, norm.ngamma = (const T*)w[9], norm.nrms = tail.rms;
  norm.dgamma = gr[10], norm.dx = k.dx_a;
  for (int64_t l = d.L - 1; l >= 0; l--) {
    Carve c{(uint8_t*)const_cast<void*>(saved), layer_bytes * (size_t)l};
    const Saved<T> s = carve_layer<T>(c, d);
    const T* x = l == 0 ? (const T*)x_ : s.x;
    Adjoint<T> a = norm;
    a.w[0] = w2 + l * D * H, a.dw[0] = gr[8] + l * D * H;                                     // w2 [D, H]
    a.x = s.g, a.part = k.part[0], a.count = 1, a.K = (int)D, a.N = (int)H;
    if (int rc = launch_adjoint<T, kNorm>(st, a, gw2)) return rc;
    a = Adjoint<T>{};
    a.w[0] = w1 + l * H * D, a.dw[0] = gr[7] + l * H * D;                                     // w1, w3 [H, D]
    a.w[1] = w3 + l * H * D, a.dw[1] = gr[9] + l * H * D;
    a.x = s.x1, a.gamma = g2 + l * D, a.rms = s.rms2;
    a.part = k.part[1], a.dots = k.dots, a.count = 2, a.K = (int)H, a.N = (int)D;
    a.in = k.part[0], a.in_bands = gw2.bands, a.h1 = s.h1, a.h3 = s.h3;
    if (int rc = launch_adjoint<T, kSwiglu>(st, a, gw13)) return rc;
    a = Adjoint<T>{};
    a.w[0] = wo + l * D * D, a.dw[0] = gr[5] + l * D * D;                                     // wo [D, D]
    a.x = s.att, a.part = k.part[0], a.count = 1, a.K = (int)D, a.N = (int)D;
    a.in = k.part[1], a.in_dots = k.dots, a.in_bands = gw13.bands, a.in_ndots = gw13.bands * gw13.cols;
    a.nx = s.x1, a.ngamma = g2 + l * D, a.nrms = s.rms2, a.residual = k.dx_a;
    a.dgamma = gr[6] + l * D, a.dx = k.dx_b;
    if (int rc = launch_adjoint<T, kNorm>(st, a, gwo)) return rc;
    const int64_t cache = l * d.pos * D;
    if (int rc = launch_llama_step_attn_bwd(st, s.q, kc + cache, vc + cache, s.k, s.v, s.att, s.lse, k.part[0], gwo.bands, gr[11] + cache,
                                            gr[12] + cache, k.dk, k.dv, k.attn, (int)d.heads, (int)d.pos, d.hd(), d.kpb_bwd(), d.scale, d.dtype))
      return rc;
    a = Adjoint<T>{};
    a.w[0] = wq + l * D * D, a.dw[0] = gr[2] + l * D * D;
    a.w[1] = wk + l * D * D, a.dw[1] = gr[3] + l * D * D;
    a.w[2] = wv + l * D * D, a.dw[2] = gr[4] + l * D * D;
    a.x = x, a.gamma = g1 + l * D, a.rms = s.rms1;
    a.part = k.part[1], a.dots = k.dots, a.count = 3, a.K = (int)D, a.N = (int)D;
    a.in = k.attn, a.in_bands = d.nsplit_bwd(), a.dk = k.dk, a.dv = k.dv;
    a.table = (const float2*)table, a.table_pairs = (int)d.table_pairs, a.head_dim = d.hd();
    if (int rc = launch_adjoint<T, kAttention>(st, a, gqkv)) return rc;
    norm = Adjoint<T>{};
    norm.in = k.part[1], norm.in_dots = k.dots, norm.in_bands = gqkv.bands, norm.in_ndots = gqkv.bands * gqkv.cols;
    norm.nx = x, norm.ngamma = g1 + l * D, norm.nrms = s.rms1, norm.residual = k.dx_b;
    norm.dgamma = gr[1] + l * D, norm.dx = k.dx_a;
  }
  norm.dx_t = gr[0], norm.K = (int)D;
  hipLaunchKernelGGL(step_norm_rows_kernel<T>, dim3((unsigned)((D + 63) / 64)), dim3(256), 0, st, norm);
  EMI_CHECK_LAUNCH("emi_llama_step_bwd(norm)");
  return EMI_OK;
}

bool dims_ok(const StepDims& d) {
  const int64_t V = d.dtype == EMI_BF16 ? 8 : 4;
  // D: the padded vector of the product kernel stands in LDS
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
