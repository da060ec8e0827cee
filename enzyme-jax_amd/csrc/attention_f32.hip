// Causal softmax attention in fp32 on the matrix cores, forward, adjoint and tangent, for gfx950:
// v_mfma_f32_16x16x4_f32 with fp32 operands and fp32 accumulation (no narrower arithmetic anywhere),
// for head_dim a multiple of 16 up to 128 and rows that start on 16-byte boundaries.  Replaces the per-head
// loop of test/llama.py:178-206 with the softmax of :13-18 for the fp32 configurations (stories15M: 6 heads x 48).
//
// A block of four (or eight) wavefronts owns 16 queries (forward, dQ; the tangent 16 or 32) or 16 keys (dK/dV). The 16-row tiles of the other sequence axis
// are dealt to the wavefronts in turn, each accumulates over its own tiles, and the partial results are added
// through the LDS at the end (the forward pass scales them to a common maximum first); that is the only barrier. A masked
// score has the weight 0 and its row is multiplied by it, so in the forward pass a NaN or an infinity in a row of v also reaches
// earlier queries of the same 16-row tile; the tangent keeps it from them (non_finite_rows). Operands come straight from global memory. What bounds it: a wavefront issues one matrix instruction per 32 cycles and its own
// 16 rows are one chain of them, so with one wavefront per 16 rows (the earlier form) the longest row set the time and too
// few wavefronts hid the loads. Causal, forward / adjoint in us: 6 heads x 256 x 48 13.6 / 40 -> 9 / 9,
// 24 heads x 1000 x 64 89 / 280 -> 56 / 161 (55 / 48 TFLOP/s), 64 heads x 2048 x 128 1329 / 4010 -> 795 / 2907 (86 / 59);
// the loads of K, V and Q through the L1 come next.
// As on the bf16 path everything is computed transposed: the score tile is S^T[other row, own row], so lane l owns row
// l % 16 for its whole life, its softmax statistics are per-lane scalars, and the probabilities leave the accumulator
// already in the B-operand layout of the second product.
//
// Operand layouts of v_mfma_f32_16x16x4_f32 (D = A . B, A 16x4, B 4x16): lane l supplies A[l % 16][l / 16] and
// B[l / 16][l % 16]; register r of lane l receives D[4 (l / 16) + r][l % 16].  The contraction index of one
// instruction is the lane group g = l / 16; which four columns (or rows) of the operand tensors the four
// groups stand for is free as long as A and B agree:
//   * products over head_dim (scores, dP): instruction (c, t) contracts columns 16 c + 4 g + t, so a lane reads
//     its row in 16-byte pieces;
//   * products over the other sequence axis (P.V, dS.K, P^T.dO, dS^T.Q): instruction t of a 16-row tile contracts
//     rows 4 g + t, which is exactly where register t of the score accumulator lives, and the output column of
//     A-row i in pass n is NT i + n (NT = head_dim / 16), so a lane reads and writes NT consecutive elements.
#include <initializer_list>
#include <stdint.h>

#include "attention_row.h"
#include "emi_device.h"

namespace emi {

typedef float f32q_t __attribute__((ext_vector_type(4)));

struct AttnShapeF32 {
  int seq, heads;
  int64_t sb, sh, ss;   // element strides of batch, head, sequence position
};

constexpr float kMasked = -1.0e30f;
// Wavefronts a block (W): 4, or 8 where few blocks have long rows: eight_forward(), eight_adjoint().
// merge_store deals the accumulator's four registers to the first four.

__device__ __forceinline__ f32q_t mfma_f32(float a, float b, f32q_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Rows row0 .. row0 + 15 (clamped to `last`) as an operand contracted over head_dim: f[c][t] of lane l is
// element (row0 + l % 16, 16 c + 4 (l / 16) + t).
template <int NT>
__device__ __forceinline__ void load_rows(const float* __restrict__ head, int64_t ss, int row0, int last, int lane,
                                          float (&f)[NT][4]) {
  int r = row0 + (lane & 15);
  r = r < last ? r : last;
  const float* p = head + (int64_t)r * ss + 4 * (lane >> 4);
#pragma unroll
  for (int c = 0; c < NT; c++) {
    const float4 x = *reinterpret_cast<const float4*>(p + 16 * c);
    f[c][0] = x.x; f[c][1] = x.y; f[c][2] = x.z; f[c][3] = x.w;
  }
}

// X . Y^T for two 16-row operands: register r of lane l is the dot product of X row 4 (l / 16) + r and Y row l % 16.
template <int NT>
__device__ __forceinline__ f32q_t rows_dot(const float (&x)[NT][4], const float (&y)[NT][4]) {
  f32q_t s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < NT; c++)
#pragma unroll
    for (int t = 0; t < 4; t++) s = mfma_f32(x[c][t], y[c][t], s);
  return s;
}

// acc += X[row0 .. row0 + 15]^T . W, where w[t] of lane l is W[row0 + 4 (l / 16) + t][l % 16] (the layout rows_dot
// leaves): acc[n][r] of lane l is output element (own row l % 16, column NT (4 (l / 16) + r) + n).  In two halves, so that
// the loads can be issued well before the weights exist.
template <int NT>
__device__ __forceinline__ void load_cols(const float* __restrict__ head, int64_t ss, int row0, int last, int lane,
                                          float (&x)[4][NT]) {
#pragma unroll
  for (int t = 0; t < 4; t++) {
    int r = row0 + 4 * (lane >> 4) + t;
    r = r < last ? r : last;                 // rows past the end carry weight 0
    const float* p = head + (int64_t)r * ss + NT * (lane & 15);
#pragma unroll
    for (int n = 0; n < NT; n++) x[t][n] = p[n];
  }
}
template <int NT>
__device__ __forceinline__ void mma_cols(const float (&x)[4][NT], const f32q_t w, f32q_t (&acc)[NT]) {
#pragma unroll
  for (int t = 0; t < 4; t++)
#pragma unroll
    for (int n = 0; n < NT; n++) acc[n] = mfma_f32(x[t][n], w[t], acc[n]);
}

// Adds the W wavefronts' accumulators and stores the sum: wavefront w < 4 takes register w of every lane, that is NT
// consecutive elements of each of the 16 rows.  `mul[i]` scales wavefront i's share.  TURN: angles are the row's (cos, sin) pairs,
// by which it is turned back (the cotangent of a vector that was rotated); a null pointer looked at instead cost the adjoint without a
// rotation 2 to 3 % (heads of 128).  The LDS is free after the next barrier.
template <int NT, int W, bool TURN = false>
__device__ __forceinline__ void merge_store(float* __restrict__ row, bool write, int lane, int wave, const f32q_t (&acc)[NT],
                                            const float (&mul)[W], float (&buf)[W][4 * NT][64], const float2* __restrict__ angles = nullptr) {
#pragma unroll
  for (int r = 0; r < 4; r++)
#pragma unroll
    for (int n = 0; n < NT; n++) buf[wave][r * NT + n][lane] = acc[n][r];
  const int first = NT * (4 * (lane >> 4) + wave);                 // this lane's first column
  [[maybe_unused]] float2 turn[NT];
  if constexpr (TURN) {
#pragma unroll
    for (int n = 0; n < NT; n++) turn[n] = wave < 4 ? angles[(first + n) >> 1] : make_float2(1.f, 0.f);
  }
  __syncthreads();
  if (W > 4 && wave >= 4) return;
  float x[NT];
#pragma unroll
  for (int n = 0; n < NT; n++) {
    x[n] = 0.f;
#pragma unroll
    for (int i = 0; i < W; i++) x[n] += buf[i][wave * NT + n][lane] * mul[i];
  }
  if constexpr (TURN) {
    float y[NT];                                                   // the pairs' other elements: with an odd NT some are other lanes'
#pragma unroll
    for (int n = 0; n < NT; n++) {
      const int e = (first + n) ^ 1, j = e / NT;
      if (NT % 2 == 0) {
        y[n] = x[n ^ 1];
      } else {
        y[n] = 0.f;
#pragma unroll
        for (int i = 0; i < W; i++) y[n] += buf[i][(j & 3) * NT + e - j * NT][(lane & 15) | ((j >> 2) << 4)] * mul[i];
      }
    }
#pragma unroll
    for (int n = 0; n < NT; n++)
      x[n] = ((first + n) & 1) == 0 ? rotated_even(turn[n].x, -turn[n].y, x[n], y[n]) : rotated_odd<float>(turn[n].x, -turn[n].y, y[n], x[n]);
  }
  if (write) {
    float* p = row + first;
#pragma unroll
    for (int n = 0; n < NT; n++) p[n] = x[n];
  }
}

// Which 16 rows and which head a block has.  Consecutive workgroups go to the eight XCDs in turn, each with an L2 of its
// own; here every XCD gets a run of whole heads, so that a head's other operands are fetched into one L2 instead of eight.
struct BlockRows { int tile, bh; };
__device__ __forceinline__ BlockRows block_rows(int tiles, int total, int id) {
  const int per = total >> 3, extra = total & 7, xcd = id & 7;
  const int w = xcd * per + (xcd < extra ? xcd : extra) + (id >> 3);
  return {w % tiles, w / tiles};
}

__device__ __forceinline__ BlockRows block_rows(int tiles) {
  return block_rows(tiles, (int)(gridDim.x * gridDim.y), (int)(blockIdx.y * gridDim.x + blockIdx.x));
}

__device__ __forceinline__ float groups_max(float x) {      // over the four lanes that share l % 16
  return max_xor32(max_xor16(x));
}
__device__ __forceinline__ float groups_sum(float x) {
  return sum_xor32(sum_xor16(x));
}

// Forward: o = softmax(scale q k^T) v, lse = log-sum-exp of the scaled scores.
template <int NT, int W>
__global__ __launch_bounds__(64 * W) void attn_fwd_f32_kernel(const float* __restrict__ q, const float* __restrict__ k,
                                                                   const float* __restrict__ v, float* __restrict__ o,
                                                                   float* __restrict__ lse, AttnShapeF32 sh, float scale,
                                                                   int causal) {
  __shared__ float buf[W][4 * NT][64];
  __shared__ float stat[2][W][16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, G = lane >> 4;
  const int tiles = (sh.seq + 15) >> 4;
  const BlockRows own = block_rows(tiles);
  const int q0 = (tiles - 1 - own.tile) * 16;                     // longest causal rows first
  const int bh = own.bh;
  const int64_t base = (int64_t)(bh / sh.heads) * sh.sb + (int64_t)(bh % sh.heads) * sh.sh;
  const int last = sh.seq - 1;
  const int myq = q0 + (lane & 15);
  float qf[NT][4];
  load_rows<NT>(q + base, sh.ss, q0, last, lane, qf);
  const int nkeys = causal ? (q0 + 16 < sh.seq ? q0 + 16 : sh.seq) : sh.seq;
  float m = kMasked, lsum = 0.f;
  f32q_t acc[NT];
#pragma unroll
  for (int n = 0; n < NT; n++) acc[n] = f32q_t{0.f, 0.f, 0.f, 0.f};
  // U key tiles per step, all their operands requested before the first product (one wait for memory per step)
  constexpr int U = NT <= 4 ? 2 : 1;
  for (int k0 = 16 * wave; k0 < nkeys; k0 += 16 * W * U) {
    f32q_t s[U];
    float kf[U][NT][4], vx[U][4][NT];
    float mx = kMasked;
#pragma unroll
    for (int u = 0; u < U; u++)
      if (k0 + 16 * W * u < nkeys) load_rows<NT>(k + base, sh.ss, k0 + 16 * W * u, last, lane, kf[u]);
#pragma unroll
    for (int u = 0; u < U; u++)
      if (k0 + 16 * W * u < nkeys) load_cols<NT>(v + base, sh.ss, k0 + 16 * W * u, last, lane, vx[u]);
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int kb = k0 + 16 * W * u;
      if (kb < nkeys) s[u] = rows_dot<NT>(kf[u], qf);
      else s[u] = f32q_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int key = kb + 4 * G + r;
        const bool valid = key < nkeys && (!causal || key <= myq);
        s[u][r] = valid ? s[u][r] * scale : kMasked;
        mx = fmaxf(mx, s[u][r]);
      }
    }
    // every tile that starts below nkeys has a key that the query sees, so the running maximum is finite from the first on
    const float m_new = fmaxf(m, groups_max(mx));
    const float alpha = expf(m - m_new);
    float psum = 0.f;
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        s[u][r] = expf(s[u][r] - m_new);
        psum += s[u][r];
      }
    lsum = lsum * alpha + psum;               // this lane's share of the row sum; the groups are added at the end
#pragma unroll
    for (int n = 0; n < NT; n++) acc[n] *= alpha;
#pragma unroll
    for (int u = 0; u < U; u++)
      if (k0 + 16 * W * u < nkeys) mma_cols<NT>(vx[u], s[u], acc);
    m = m_new;
  }
  lsum = groups_sum(lsum);
  if (G == 0) {
    stat[0][wave][lane] = m;
    stat[1][wave][lane] = lsum;
  }
  __syncthreads();
  float mul[W], top = kMasked, sum = 0.f;
#pragma unroll
  for (int i = 0; i < W; i++) top = fmaxf(top, stat[0][i][lane & 15]);     // wavefront 0 has key 0: finite
#pragma unroll
  for (int i = 0; i < W; i++) {
    mul[i] = expf(stat[0][i][lane & 15] - top);                                 // 0 for a wavefront without a tile
    sum += stat[1][i][lane & 15] * mul[i];
  }
#pragma unroll
  for (int i = 0; i < W; i++) mul[i] *= 1.f / sum;
  merge_store<NT, W>(o + base + (int64_t)myq * sh.ss, myq < sh.seq, lane, wave, acc, mul, buf);
  if (wave == 0 && G == 0 && myq < sh.seq) lse[(int64_t)bh * sh.seq + myq] = top + logf(sum);
}

// dV = P^T dO, dK = scale dS^T Q: a block per 16 keys, walking the queries that see them.
// DELTA: from the rows of o, where nothing has left delta.
template <int NT, int W, bool DELTA, bool TURN>
__device__ __forceinline__ void bwd_dkv_rows(const BlockRows own, const float* __restrict__ q, const float* __restrict__ k,
                                             const float* __restrict__ v, const float* __restrict__ o, const float* __restrict__ d_o,
                                             const float* __restrict__ lse, const float* __restrict__ delta, float* __restrict__ dk,
                                             float* __restrict__ dv, AttnShapeF32 sh, float scale, int causal,
                                             const float2* __restrict__ unrope, float (&buf)[W][4 * NT][64]) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, G = lane >> 4;
  const int key0 = own.tile * 16;                                  // the earliest keys see the most queries
  const int bh = own.bh;
  const int64_t base = (int64_t)(bh / sh.heads) * sh.sb + (int64_t)(bh % sh.heads) * sh.sh;
  const int last = sh.seq - 1;
  const int mykey = key0 + (lane & 15);
  float kf[NT][4], vf[NT][4];
  load_rows<NT>(k + base, sh.ss, key0, last, lane, kf);
  load_rows<NT>(v + base, sh.ss, key0, last, lane, vf);
  const float* lrow = lse + (int64_t)bh * sh.seq;
  [[maybe_unused]] const float* drow = DELTA ? nullptr : delta + (int64_t)bh * sh.seq;
  f32q_t acck[NT], accv[NT];
#pragma unroll
  for (int n = 0; n < NT; n++) acck[n] = accv[n] = f32q_t{0.f, 0.f, 0.f, 0.f};
  for (int qb = (causal ? key0 : 0) + 16 * wave; qb < sh.seq; qb += 16 * W) {
    float qf[NT][4], dof[NT][4], qx[4][NT], dox[4][NT], lq[4], dq_[4];
    load_rows<NT>(q + base, sh.ss, qb, last, lane, qf);
    load_rows<NT>(d_o + base, sh.ss, qb, last, lane, dof);
    load_cols<NT>(d_o + base, sh.ss, qb, last, lane, dox);    // for dV += P^T . dO
    load_cols<NT>(q + base, sh.ss, qb, last, lane, qx);       // for dK += dS^T . Q
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int qi = qb + 4 * G + r;
      const int qc = qi < last ? qi : last;
      lq[r] = lrow[qc];
      if constexpr (!DELTA) dq_[r] = drow[qc];
    }
    if constexpr (DELTA) {
      float of[NT][4], dl = 0.f;
      load_rows<NT>(o + base, sh.ss, qb, last, lane, of);
#pragma unroll
      for (int c = 0; c < NT; c++)
#pragma unroll
        for (int t = 0; t < 4; t++) dl += of[c][t] * dof[c][t];
      dl = groups_sum(dl);                              // of query qb + l % 16
#pragma unroll
      for (int r = 0; r < 4; r++) dq_[r] = __shfl(dl, 4 * G + r);
    }
    f32q_t s = rows_dot<NT>(qf, kf);                   // register r: query qb + 4 G + r, key mykey
    f32q_t dp = rows_dot<NT>(dof, vf);
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int qi = qb + 4 * G + r;
      const bool valid = qi < sh.seq && (!causal || mykey <= qi);
      const float p = valid ? expf(s[r] * scale - lq[r]) : 0.f;
      s[r] = p;
      dp[r] = p * (dp[r] - dq_[r]) * scale;
    }
    mma_cols<NT>(dox, s, accv);
    mma_cols<NT>(qx, dp, acck);
  }
  float one[W];
#pragma unroll
  for (int i = 0; i < W; i++) one[i] = 1.f;
  merge_store<NT, W, TURN>(dk + base + (int64_t)mykey * sh.ss, mykey < sh.seq, lane, wave, acck, one, buf,
                           TURN ? unrope + (int64_t)(mykey < last ? mykey : last) * (8 * NT) : nullptr);
  __syncthreads();
  merge_store<NT, W>(dv + base + (int64_t)mykey * sh.ss, mykey < sh.seq, lane, wave, accv, one, buf);
}

template <int NT, int W, bool TURN>
__global__ __launch_bounds__(64 * W) void attn_bwd_dkv_f32_kernel(const float* __restrict__ q, const float* __restrict__ k,
                                                                       const float* __restrict__ v,
                                                                       const float* __restrict__ d_o,
                                                                       const float* __restrict__ lse,
                                                                       const float* __restrict__ delta, float* __restrict__ dk,
                                                                       float* __restrict__ dv, AttnShapeF32 sh, float scale,
                                                                       int causal, const float2* __restrict__ unrope) {
  __shared__ float buf[W][4 * NT][64];
  bwd_dkv_rows<NT, W, false, TURN>(block_rows((sh.seq + 15) >> 4), q, k, v, nullptr, d_o, lse, delta, dk, dv, sh, scale, causal, unrope, buf);
}

// dQ = scale dS K with dS = P (dP - delta), P = exp(scale q k^T - lse), dP = dO V^T, delta = rowsum(dO * O), which it also
// leaves for the dK/dV kernel.
// BOTH: one launch (grid.z: 0 dK/dV, 1 dQ) for sequences and heads that leave the chip half empty: the two run side by side
// instead of one after the other, and dK/dV forms delta itself.
// dQ stands in its kernel, dK/dV in a function of its own: the order of the loads that the compiler makes of either depends
// on that.  us, dQ in a function | here: 24 heads x 1000 x 96 261 | 247, 8 x 3000 x 128 784 | 768; dK/dV in its kernel | in a
// function: 24 x 1000 x 32 105 | 98, 64 x 1024 x 48 294 | 284.
template <int NT, int W, bool BOTH, bool TURN>
__global__ __launch_bounds__(64 * W) void attn_bwd_dq_f32_kernel(const float* __restrict__ q, const float* __restrict__ k,
                                                                      const float* __restrict__ v, const float* __restrict__ o,
                                                                      const float* __restrict__ d_o,
                                                                      const float* __restrict__ lse, float* __restrict__ delta,
                                                                      float* __restrict__ dq, float* __restrict__ dk,
                                                                      float* __restrict__ dv, AttnShapeF32 sh, float scale,
                                                                      int causal, const float2* __restrict__ unrope) {
  __shared__ float buf[W][4 * NT][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, G = lane >> 4;
  const int tiles = (sh.seq + 15) >> 4;
  const BlockRows own = block_rows(tiles);
  if constexpr (BOTH) {
    if (blockIdx.z == 0) {
      bwd_dkv_rows<NT, W, true, TURN>(own, q, k, v, o, d_o, lse, nullptr, dk, dv, sh, scale, causal, unrope, buf);
      return;
    }
  }
  const int q0 = (tiles - 1 - own.tile) * 16;
  const int bh = own.bh;
  const int64_t base = (int64_t)(bh / sh.heads) * sh.sb + (int64_t)(bh % sh.heads) * sh.sh;
  const int last = sh.seq - 1;
  const int myq = q0 + (lane & 15);
  const int qc = myq < last ? myq : last;
  float qf[NT][4], dof[NT][4];
  load_rows<NT>(q + base, sh.ss, q0, last, lane, qf);
  load_rows<NT>(d_o + base, sh.ss, q0, last, lane, dof);
  const float L = lse[(int64_t)bh * sh.seq + qc];
  float dl = 0.f;
  {
    float of[NT][4];
    load_rows<NT>(o + base, sh.ss, q0, last, lane, of);
#pragma unroll
    for (int c = 0; c < NT; c++)
#pragma unroll
      for (int t = 0; t < 4; t++) dl += of[c][t] * dof[c][t];
    dl = groups_sum(dl);
    if (!BOTH && wave == 0 && G == 0 && myq < sh.seq) delta[(int64_t)bh * sh.seq + myq] = dl;
  }
  const int nkeys = causal ? (q0 + 16 < sh.seq ? q0 + 16 : sh.seq) : sh.seq;
  f32q_t acc[NT];
#pragma unroll
  for (int n = 0; n < NT; n++) acc[n] = f32q_t{0.f, 0.f, 0.f, 0.f};
  for (int kb = 16 * wave; kb < nkeys; kb += 16 * W) {
    float kf[NT][4], vf[NT][4], kx[4][NT];
    load_rows<NT>(k + base, sh.ss, kb, last, lane, kf);
    load_rows<NT>(v + base, sh.ss, kb, last, lane, vf);
    load_cols<NT>(k + base, sh.ss, kb, last, lane, kx);        // for dQ += dS . K
    f32q_t s = rows_dot<NT>(kf, qf);
    const f32q_t dp = rows_dot<NT>(vf, dof);
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int key = kb + 4 * G + r;
      const bool valid = key < nkeys && (!causal || key <= myq);
      const float p = valid ? expf(s[r] * scale - L) : 0.f;
      s[r] = p * (dp[r] - dl) * scale;
    }
    mma_cols<NT>(kx, s, acc);
  }
  float one[W];
#pragma unroll
  for (int i = 0; i < W; i++) one[i] = 1.f;
  merge_store<NT, W, TURN>(dq + base + (int64_t)myq * sh.ss, myq < sh.seq, lane, wave, acc, one, buf,
                           TURN ? unrope + (int64_t)qc * (8 * NT) : nullptr);
}

// Where a row of v or tv that not all queries of a block see is not finite, the masked weight 0 would carry it to the others, as it
// would those that stand in for rows past the end: the tangent's block works such queries out row by row.  It looks at these rows beside
// the loads of q where the CU has another block meanwhile, and otherwise once they are in registers, in the last tile of
// one or two wavefronts.  us, neither | before | after, causal heads x length x head size: 32 x 512 x 48 69 | 68 | 71, 32 x 1716 x 64 547 |
// 540 | 546, 32 x 512 x 80 106 | 107 | 111; 32 x 512 x 96 123 | 128 | 122, 32 x 1716 x 96 826 | 867 | 804, 32 x 1716 x 128 1107 | 1121 | 1108.
//
// A NaN in one of the block's threads if the rows row0 .. end - 1 of a head (at most 16) hold a NaN or an infinity.
template <int NT>
__device__ __forceinline__ float non_finite_rows(const float* __restrict__ head, int64_t ss, int row0, int end) {
  float z = 0.f;
#pragma unroll
  for (int u = 0; u < (NT + 3) / 4; u++) {
    const int i = u * 256 + (int)threadIdx.x, r = row0 + i / (4 * NT);
    const float4 x = *reinterpret_cast<const float4*>(head + (int64_t)(r < end ? r : end - 1) * ss + 4 * (i % (4 * NT)));
    z = fmaf(x.x, 0.f, fmaf(x.y, 0.f, fmaf(x.z, 0.f, fmaf(x.w, 0.f, z))));
  }
  return z;
}

// A NaN if one of the values is a NaN or an infinity.
template <int NT> __device__ __forceinline__ float non_finite(const float (&x)[4][NT]) {
  float z = 0.f;
#pragma unroll
  for (int t = 0; t < 4; t++)
#pragma unroll
    for (int n = 0; n < NT; n++) z = fmaf(x[t][n], 0.f, z);
  return z;
}

// Tangent: with p = exp(scale q k^T - lse) and tS = scale (tq k^T + q tk^T)
//   to = sum_j p_j tv_j + sum_j p_j tS_j v_j - mu o,   o = sum_j p_j v_j,   mu = sum_j p_j tS_j
// in one walk over the keys: six products, and two accumulators (the first two sums are one).  QS sets of 16 queries share every
// row of K, V, tK and tV that is loaded.  A null tangent skips its loads and products.  What bounds it: as above, and from heads
// of 96 on one wavefront a SIMD (of 128: 322 registers with one set of queries, 500 with two).  Causal, us, a wavefront per query without matrix instructions | this: 16 heads x
// 1122 x 64 3918 | 103, 32 x 1716 x 64 16918 | 405 (89 TFLOP/s), 96 x 1817 x 128 117047 | 2662 (91), 6 x 256 x 48 143 | 10;
// error against float64 4.7e-7 | 4.2e-7 at 32 x 512 x 128.
template <int NT, int QS>
__global__ __launch_bounds__(64 * 4) void attn_jvp_f32_kernel(const float* __restrict__ q, const float* __restrict__ k,
                                                                   const float* __restrict__ v, const float* __restrict__ lse,
                                                                   const float* __restrict__ tq, const float* __restrict__ tk,
                                                                   const float* __restrict__ tv, float* __restrict__ to,
                                                                   AttnShapeF32 sh, float scale, int causal) {
  __shared__ float buf[4][4 * NT][64];
  __shared__ float stat[QS][4][16];
  __shared__ int by_row[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, G = lane >> 4;
  const int tiles = (sh.seq + 16 * QS - 1) / (16 * QS);
  const BlockRows own = block_rows(tiles);
  const int q0 = (tiles - 1 - own.tile) * 16 * QS;                // longest causal rows first
  const int bh = own.bh;
  const int64_t base = (int64_t)(bh / sh.heads) * sh.sb + (int64_t)(bh % sh.heads) * sh.sh;
  const int last = sh.seq - 1;
  float qf[QS][NT][4], tqf[QS][NT][4], L[QS], mu[QS];
  f32q_t acct[QS][NT], acco[QS][NT];
#pragma unroll
  for (int s = 0; s < QS; s++) {
    load_rows<NT>(q + base, sh.ss, q0 + 16 * s, last, lane, qf[s]);
    if (tq != nullptr) load_rows<NT>(tq + base, sh.ss, q0 + 16 * s, last, lane, tqf[s]);
    const int myq = q0 + 16 * s + (lane & 15);
    L[s] = lse[(int64_t)bh * sh.seq + (myq < last ? myq : last)];
    mu[s] = 0.f;
#pragma unroll
    for (int n = 0; n < NT; n++) acct[s][n] = acco[s][n] = f32q_t{0.f, 0.f, 0.f, 0.f};
  }
  const int nkeys = causal ? (q0 + 16 * QS < sh.seq ? q0 + 16 * QS : sh.seq) : sh.seq;
  auto tile = [&](int kb, float (&vx)[4][NT], float (&tvx)[4][NT]) __attribute__((always_inline)) {
    float kf[NT][4], tkf[NT][4];
    load_rows<NT>(k + base, sh.ss, kb, last, lane, kf);
    if (tk != nullptr) load_rows<NT>(tk + base, sh.ss, kb, last, lane, tkf);
    load_cols<NT>(v + base, sh.ss, kb, last, lane, vx);
    if (tv != nullptr) load_cols<NT>(tv + base, sh.ss, kb, last, lane, tvx);
#pragma unroll
    for (int s = 0; s < QS; s++) {
      const int myq = q0 + 16 * s + (lane & 15);
      f32q_t p = rows_dot<NT>(kf, qf[s]);
      f32q_t w = f32q_t{0.f, 0.f, 0.f, 0.f}, w2 = w;
      if (tq != nullptr) w = rows_dot<NT>(kf, tqf[s]);
      if (tk != nullptr) w2 = rows_dot<NT>(tkf, qf[s]);
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int key = kb + 4 * G + r;
        const bool valid = key < nkeys && (!causal || key <= myq);
        p[r] = valid ? expf(p[r] * scale - L[s]) : 0.f;
        w[r] = valid ? p[r] * (w[r] + w2[r]) * scale : 0.f;
        mu[s] += w[r];
      }
      mma_cols<NT>(vx, p, acco[s]);
      mma_cols<NT>(vx, w, acct[s]);
      if (tv != nullptr) mma_cols<NT>(tvx, p, acct[s]);
    }
  };
  int odd = 0;
  if constexpr (QS == 1 && NT <= 5) {                              // two or more wavefronts a SIMD
    float z = non_finite_rows<NT>(v + base, sh.ss, causal ? q0 : last, nkeys);
    if (tv != nullptr) z += non_finite_rows<NT>(tv + base, sh.ss, causal ? q0 : last, nkeys);
    odd = __any(z != 0.f);                                         // (NaN)
    if (lane == 0) by_row[wave] = odd;
    for (int kb = 16 * wave; kb < nkeys; kb += 16 * 4) {
      float vx[4][NT], tvx[4][NT];
      tile(kb, vx, tvx);
    }
  } else {
    float vx[4][NT], tvx[4][NT];
    int kb = 16 * wave;
    for (; kb < nkeys; kb += 16 * 4) tile(kb, vx, tvx);
    kb -= 16 * 4;
    if (kb >= 0 && kb + 15 > (causal ? q0 : last)) odd = __any(non_finite<NT>(vx) + (tv != nullptr ? non_finite<NT>(tvx) : 0.f) != 0.f);
    if (lane == 0) by_row[wave] = odd;
  }
#pragma unroll
  for (int s = 0; s < QS; s++) {
    mu[s] = groups_sum(mu[s]);
    if (G == 0) stat[s][wave][lane] = mu[s];
  }
  __syncthreads();
  const float one[4] = {1.f, 1.f, 1.f, 1.f};
#pragma unroll
  for (int s = 0; s < QS; s++) {
    float m = 0.f;
#pragma unroll
    for (int i = 0; i < 4; i++) m += stat[s][i][lane & 15];
#pragma unroll
    for (int n = 0; n < NT; n++) acct[s][n] -= m * acco[s][n];
    const int myq = q0 + 16 * s + (lane & 15);
    if (s > 0) __syncthreads();                                    // buf has been read
    merge_store<NT, 4>(to + base + (int64_t)myq * sh.ss, myq < sh.seq, lane, wave, acct[s], one, buf);
  }
  if (by_row[0] | by_row[1] | by_row[2] | by_row[3]) {
    __syncthreads();                                               // the rows have been stored
    for (int qi = q0 + wave; qi < q0 + 16 * QS && qi < sh.seq; qi += 4)
      attn_jvp_row<float>(q, k, v, lse[(int64_t)bh * sh.seq + qi], tq, tk, tv, to, qi, causal ? qi + 1 : sh.seq, {base, sh.ss, 16 * NT, lane, scale});
  }
}

bool attn_f32_mfma_ok(int64_t seq, int64_t d, int64_t sb, int64_t shh, int64_t ss, std::initializer_list<const void*> ptrs) {
  if (d % 16 != 0 || d > 128 || seq < 1) return false;
  if ((sb | shh | ss) & 3) return false;
  for (const void* p : ptrs)
    if (reinterpret_cast<uintptr_t>(p) & 15) return false;
  return true;
}

// Eight wavefronts a block where the blocks have a CU each and the longest row, which sets the time, is of tiles enough; heads of
// 64 and rows without a mask fill the matrix cores sooner.  us, four | eight, heads x length x head size (blocks): forward, causal
// 6 x 256 x 48 (96) 6.5 | 6.3, 6 x 512 x 48 (192) 10.0 | 8.9, 8 x 400 x 64 (200) 10.1 | 9.9, 6 x 128 x 48 (48) 4.7 | 5.2, 24 x 200 x 48 (312)
// 7.0 | 8.1; adjoint (one launch), causal 6 x 256 x 48 9.8 | 8.8, 12 x 200 x 48 (156) 11.2 | 9.3, 6 x 512 x 48 19.6 | 14.8, 8 x 512 x 64 (256)
// 29.5 | 25.1, 24 x 128 x 48 (192) 7.9 | 8.4, 12 x 256 x 64 (192) 16.4 | 18.2; all keys 8 x 256 x 48 (128) 10.2 | 9.2, 8 x 512 x 48 22.1 | 23.3.
static bool eight_forward(int64_t blocks, int64_t seq, int64_t head_dim, int causal) {
  return head_dim <= 64 && blocks <= 256 && seq >= (head_dim <= 48 && causal ? 192 : 384);
}
// In the adjoint with heads of 48 and 64 a CU has room for one such block, and an XCD's run of rows is of two rounds of them from 160
// blocks on: dQ's long rows come too late there unless they are the first of the run, which is a head then or a part of one.  us, four |
// eight, forward and adjoint, heads of 48: 8 x 384 (192 blocks) 26.9 | 24.1, 6 x 640 (240) 39.1 | 35.4, 8 x 448 (224) 29.9 | 26.0, 2 x 2000 (250) 92 |
// 87, but 14 x 256 (224) 22.0 | 23.3, 10 x 384 (240) 28.4 | 30.2, 9 x 448 (252) 28.8 | 32.0, 3 x 1300 (246) 61 | 66; of 64: 8 x 512 (256) 43.9 |
// 39.4, 10 x 384 37.0 | 40.8, 5 x 800 (250) 55.7 | 58.5.  Heads of 32, two such blocks a CU: 9 x 448 28.0 | 26.5, 3 x 1300 55 | 50.
static bool eight_adjoint(int64_t blocks, int64_t heads, int64_t seq, int64_t head_dim, int causal) {
  const bool long_first = head_dim <= 32 || blocks <= 160 || (heads >= 6 && heads <= 8) || 8 % heads == 0;
  if (head_dim > 48) return head_dim <= 64 && causal && seq >= 384 && blocks <= 256 && long_first;
  return seq >= 96 && (causal ? blocks <= 160 || (seq >= 256 && blocks <= 256 && long_first) : blocks <= 128);
}

#define EMI_ATTN_F32_DISPATCH(NTV, CALL)      \
  switch (NTV) {                              \
    case 1: { constexpr int NT = 1; CALL; break; } \
    case 2: { constexpr int NT = 2; CALL; break; } \
    case 3: { constexpr int NT = 3; CALL; break; } \
    case 4: { constexpr int NT = 4; CALL; break; } \
    case 5: { constexpr int NT = 5; CALL; break; } \
    case 6: { constexpr int NT = 6; CALL; break; } \
    case 7: { constexpr int NT = 7; CALL; break; } \
    default: { constexpr int NT = 8; CALL; break; } \
  }

// Forward on the fp32 matrix-core path; -1 when the operands do not qualify (the caller then takes the
// one-wavefront-per-row kernel).
int launch_attn_fwd_f32_mfma(hipStream_t st, const void* q, const void* k, const void* v, void* o, float* lse, int64_t batch,
                             int64_t heads, int64_t seq, int64_t head_dim, int64_t sb, int64_t shh, int64_t ss, float scale,
                             int causal) {
  if (!attn_f32_mfma_ok(seq, head_dim, sb, shh, ss, {q, k, v, o})) return -1;
  const AttnShapeF32 shp{(int)seq, (int)heads, sb, shh, ss};
  const dim3 grid((unsigned)((seq + 15) / 16), (unsigned)(batch * heads));
#define EMI_FWD(W)                                                                                                                   \
  EMI_ATTN_F32_DISPATCH((int)(head_dim / 16),                                                                                        \
                        hipLaunchKernelGGL((attn_fwd_f32_kernel<(W == 8 && NT > 4 ? 4 : NT), W>), grid, dim3(64 * W), 0, st, (const float*)q, \
                                           (const float*)k, (const float*)v, (float*)o, lse, shp, scale, causal))
  if (eight_forward((int64_t)grid.x * grid.y, seq, head_dim, causal)) EMI_FWD(8)
  else EMI_FWD(4)
#undef EMI_FWD
  EMI_CHECK_LAUNCH("emi_attn_fwd(fp32 mfma)");
  return EMI_OK;
}

template <bool TURN>
static int launch_bwd(hipStream_t st, const void* q, const void* k, const void* v, const void* o, const void* d_o, const float* lse, float* delta,
                      void* dq, void* dk, void* dv, int64_t batch, int64_t heads, int64_t seq, int64_t head_dim, int64_t sb, int64_t shh, int64_t ss,
                      float scale, int causal, const float2* angles) {
  const AttnShapeF32 shp{(int)seq, (int)heads, sb, shh, ss};
  const dim3 grid((unsigned)((seq + 15) / 16), (unsigned)(batch * heads));
  // One launch while two would each leave much of the chip idle, up to `most` blocks.  Of causal rows the late ones are the
  // longest and end alone, so that the other kernel's blocks find room; with rows of more than 1024 there are too few of them,
  // and without the mask all blocks end together and the one launch gains only while it is small.  Heads of 128 take 188
  // registers in the one launch (dQ those of dK/dV), one block a CU, where the two have two and three.
  // us, two | one, heads x length x head size (blocks): causal 6 x 256 x 48 (96) 14.7 | 9.2, 24 x 512 x 48 (768) 54 | 37,
  // 24 x 512 x 64 (768) 72 | 59, 32 x 512 x 64 (1024) 1.16 times, 256 x 64 x 64 (1024) 0.96, 8 x 2048 x 64 (1024) 0.95,
  // 6 x 2000 x 48 (750) 0.90, 8 x 1000 x 96 (504) 110 | 86, 12 x 512 x 128 (384) 1.25, 64 x 128 x 128 (512) 38 | 43,
  // 4 x 2000 x 128 (500) 0.84; all keys 12 x 777 x 48 (588) 1.11, 128 x 128 x 48 (1024) 1.09, 12 x 1000 x 32 (756) 0.84,
  // 64 x 128 x 96 (512) 1.04, 8 x 1000 x 96 (504) 139 | 149, 6 x 500 x 128 (192) 0.93, 8 x 1000 x 128 (504) 179 | 240.
  const bool middling = seq >= 192 && seq <= 1024;
  int64_t most;
  if (!causal) most = head_dim <= 48 ? (seq < 512 ? 1024 : 640) : head_dim <= 112 ? (seq < 256 ? 512 : 448) : 128;
  else if (head_dim <= 48) most = seq <= 1024 ? 1024 : 512;
  else if (head_dim <= 64) most = middling ? 1024 : 512;
  else most = head_dim <= 112 || middling ? 512 : 192;
  if ((int64_t)grid.x * grid.y <= most) {
#define EMI_BOTH(W)                                                                                                                      \
  EMI_ATTN_F32_DISPATCH((int)(head_dim / 16),                                                                                            \
                        hipLaunchKernelGGL((attn_bwd_dq_f32_kernel<(W == 8 && NT > 4 ? 4 : NT), W, true, TURN>), dim3(grid.x, grid.y, 2), dim3(64 * W), 0, \
                                           st, (const float*)q, (const float*)k, (const float*)v, (const float*)o, (const float*)d_o, lse, \
                                           nullptr, (float*)dq, (float*)dk, (float*)dv, shp, scale, causal, angles))
    if (eight_adjoint((int64_t)grid.x * grid.y, grid.y, seq, head_dim, causal)) EMI_BOTH(8)
    else EMI_BOTH(4)
#undef EMI_BOTH
    EMI_CHECK_LAUNCH("emi_attn_bwd(fp32 mfma)");
    return EMI_OK;
  }
  EMI_ATTN_F32_DISPATCH((int)(head_dim / 16),
                        hipLaunchKernelGGL((attn_bwd_dq_f32_kernel<NT, 4, false, TURN>), grid, dim3(256), 0, st, (const float*)q,
                                           (const float*)k, (const float*)v, (const float*)o, (const float*)d_o, lse, delta,
                                           (float*)dq, nullptr, nullptr, shp, scale, causal, angles));
  EMI_CHECK_LAUNCH("emi_attn_bwd(fp32 mfma dq)");
  EMI_ATTN_F32_DISPATCH((int)(head_dim / 16),
                        hipLaunchKernelGGL((attn_bwd_dkv_f32_kernel<NT, 4, TURN>), grid, dim3(256), 0, st, (const float*)q,
                                           (const float*)k, (const float*)v, (const float*)d_o, lse, delta, (float*)dk,
                                           (float*)dv, shp, scale, causal, angles));
  EMI_CHECK_LAUNCH("emi_attn_bwd(fp32 mfma dkv)");
  return EMI_OK;
}

// dQ, dK, dV on the fp32 matrix-core path (delta: scratch for rowsum(dO * O); unrope: null, or the table by which dq and dk are
// turned back); -1 when the operands do not qualify.
int launch_attn_bwd_f32_mfma(hipStream_t st, const void* q, const void* k, const void* v, const void* o, const void* d_o,
                             const float* lse, float* delta, void* dq, void* dk, void* dv, int64_t batch, int64_t heads,
                             int64_t seq, int64_t head_dim, int64_t sb, int64_t shh, int64_t ss, float scale, int causal,
                             const float* unrope) {
  if (!attn_f32_mfma_ok(seq, head_dim, sb, shh, ss, {q, k, v, o, d_o, dq, dk, dv})) return -1;
  const float2* angles = reinterpret_cast<const float2*>(unrope);
  return angles == nullptr ? launch_bwd<false>(st, q, k, v, o, d_o, lse, delta, dq, dk, dv, batch, heads, seq, head_dim, sb, shh, ss, scale, causal, angles)
                           : launch_bwd<true>(st, q, k, v, o, d_o, lse, delta, dq, dk, dv, batch, heads, seq, head_dim, sb, shh, ss, scale, causal, angles);
}

// Tangent on the fp32 matrix-core path (null tangents: zero); -1 when the operands do not qualify.
int launch_attn_jvp_f32_mfma(hipStream_t st, const void* q, const void* k, const void* v, const float* lse, const void* tq,
                             const void* tk, const void* tv, void* to, int64_t batch, int64_t heads, int64_t seq, int64_t head_dim,
                             int64_t sb, int64_t shh, int64_t ss, float scale, int causal) {
  if (!attn_f32_mfma_ok(seq, head_dim, sb, shh, ss, {q, k, v, tq, tk, tv, to})) return -1;
  const AttnShapeF32 shp{(int)seq, (int)heads, sb, shh, ss};
#define EMI_JVP_F32(QS)                                                                                                         \
  do {                                                                                                                          \
    const dim3 grid((unsigned)((seq + 16 * QS - 1) / (16 * QS)), (unsigned)(batch * heads));                                    \
    EMI_ATTN_F32_DISPATCH((int)(head_dim / 16),                                                                                 \
                          hipLaunchKernelGGL((attn_jvp_f32_kernel<NT, QS>), grid, dim3(64 * 4), 0, st, (const float*)q,    \
                                             (const float*)k, (const float*)v, lse, (const float*)tq, (const float*)tk,         \
                                             (const float*)tv, (float*)to, shp, scale, causal));                                \
  } while (0)
  // Two sets a block where the rows are long enough that their loads count and there are blocks enough; a causal block of 32
  // queries multiplies more masked keys, and the long ones end alone.  us, one set | two, heads x length x head size: causal
  // 32 x 2048 x 128 1360 | 1105, 32 x 777 x 128 235 | 199, 32 x 500 x 128 104 | 122, 8 x 1500 x 128 210 | 191, 8 x 1000 x 128
  // 90 | 129, 128 x 500 x 80 221 | 236, 32 x 1500 x 80 404 | 375, 32 x 2048 x 64 528 | 551; all keys 32 x 1000 x 96 498 | 387,
  // 8 x 777 x 128 132 | 108, 8 x 500 x 128 45 | 68.
  const int64_t pairs = (seq + 31) / 32 * batch * heads;
  if (head_dim >= 80 && (causal ? seq > 512 && pairs > 320 : pairs >= 200)) EMI_JVP_F32(2);
  else EMI_JVP_F32(1);
#undef EMI_JVP_F32
  EMI_CHECK_LAUNCH("emi_attn_jvp(fp32 mfma)");
  return EMI_OK;
}

}  // namespace emi
