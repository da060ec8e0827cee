// The tangent of one causal or full softmax attention row by one wavefront, for the kernels that work row by row.
#pragma once
#include "emi_device.h"

namespace emi {

struct AttnRowTangent {                            // operands of one (batch, head): rows `ss` elements apart
  int64_t base, ss;
  int d, lane;
  float scale;
};

// tS = scale (tq k^T + q tk^T);  to = sum_j p_j tS_j v_j - (sum_j p_j tS_j) o + sum_j p_j tv_j over the keys 0 .. nkeys - 1,
// p_j = exp(S_j - L).  Rows of v and tv behind nkeys are not read.  One key per lane and 64 keys per sweep; d <= 256.
template <typename T>
__device__ __forceinline__ void attn_jvp_row(const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v, float L,
                                             const T* __restrict__ tq, const T* __restrict__ tk, const T* __restrict__ tv, T* __restrict__ to,
                                             int qi, int nkeys, const AttnRowTangent& a) {
  const int64_t base = a.base;
  const int lane = a.lane, d = a.d;
  const float scale = a.scale;
  const T* qr = q + base + (int64_t)qi * a.ss;
  const T* tqr = tq ? tq + base + (int64_t)qi * a.ss : nullptr;
  float mu = 0.f;
  float acc_w[4] = {0.f, 0.f, 0.f, 0.f}, acc_o[4] = {0.f, 0.f, 0.f, 0.f}, acc_t[4] = {0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < nkeys; k0 += 64) {
    const int key = k0 + lane;
    float p = 0.f, w = 0.f;
    if (key < nkeys) {
      const T* kr = k + base + (int64_t)key * a.ss;
      const T* tkr = tk ? tk + base + (int64_t)key * a.ss : nullptr;
      float s = 0.f, ts = 0.f;
      for (int i = 0; i < d; i++) {
        const float qv = to_f32(qr[i]), kv = to_f32(kr[i]);
        s = fmaf(qv, kv, s);
        if (tqr) ts = fmaf(to_f32(tqr[i]), kv, ts);
        if (tkr) ts = fmaf(qv, to_f32(tkr[i]), ts);
      }
      p = expf(s * scale - L);
      w = p * ts * scale;
    }
    mu += wave_sum(w);
    const int cnt = nkeys - k0 < 64 ? nkeys - k0 : 64;
    for (int j = 0; j < cnt; j++) {
      const float pj = __shfl(p, j, 64), wj = __shfl(w, j, 64);
      const T* vr = v + base + (int64_t)(k0 + j) * a.ss;
      const T* tvr = tv ? tv + base + (int64_t)(k0 + j) * a.ss : nullptr;
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const int i = lane + c * 64;
        if (i < d) {
          const float vv = to_f32(vr[i]);
          acc_w[c] = fmaf(wj, vv, acc_w[c]);
          acc_o[c] = fmaf(pj, vv, acc_o[c]);
          if (tvr) acc_t[c] = fmaf(pj, to_f32(tvr[i]), acc_t[c]);
        }
      }
    }
  }
  T* out = to + base + (int64_t)qi * a.ss;
#pragma unroll
  for (int c = 0; c < 4; c++) {
    const int i = lane + c * 64;
    if (i < d) out[i] = from_f32<T>(acc_w[c] - mu * acc_o[c] + acc_t[c]);
  }
}

}  // namespace emi
