// Decoder layers over whole sequences (test/llama.py:144-233, batched and causal) as one call each way: forward through L
// layers whose weights are stacked, and the reverse pass with every gradient.
//
// No kernel of its own: it issues the launchers of emi.h in the order in which ops.attention_block, ops.ffn and their rules
// do.  A layer is seven to twelve launches forward and about twenty in reverse, and a small model's are 3 to 10 us each, less
// than a Python operator costs: the dim-288 model on 256 tokens spent 2.6 ms on the host for 1.25 ms of kernels.
// The rotation of q and k, the SwiGLU and its adjoint are part of the products before them where that is faster (gemm_tail):
// bf16 layer forward 68 -> 56 us at dim 768 on 777 tokens, 131 -> 116 at dim 1024 on 2000; fp32 50 -> 46 at dim 288 on 200.
// In reverse the weight gradients dW = dY^T X feed nothing else, so they wait until `group` layers are done and run grouped
// by shape (q, k, v, o; w1, w3; w2), which fills the chip where one layer's would not; a group of one runs them in place.
// So do the column sums of the RMSNorm adjoints (dim-288 model, six layers: 11 launches of 3 us less, 858 -> 830 us).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/emi.h"
#include "gemm_plan.h"
#include "rmsnorm.h"

extern "C" int emi_fail(int code, const char* fmt, ...);

namespace {

enum { kAtt, kQ, kK, kV, kO, kFfn, kW1, kW2, kW3, kWeights };      // the order of the stacked weights

struct Dims {
  int64_t L, B, S, D, H, heads;
  float eps, scale;
  int dtype;
  int64_t T() const { return B * S; }
  int64_t hd() const { return D / heads; }
  size_t elt() const { return dtype == EMI_BF16 ? 2 : 4; }
  bool ok() const {
    return L > 0 && B > 0 && S > 0 && D > 0 && H > 0 && heads > 0 && D % heads == 0 && hd() % 2 == 0 && D % 8 == 0 && H % 8 == 0 &&
           (dtype == EMI_F32 || dtype == EMI_BF16) && T() > 8;
  }
  bool tiles(int64_t n) const { return T() % 256 == 0 && n % 256 == 0 && (T() / 256) * (n / 256) >= 192; }
  // the kernels with RoPE in their epilogues (ops.attention_block)
  bool rope_attention() const { return dtype == EMI_BF16 && (hd() == 64 || hd() == 128) && S >= 128; }
  // the adjoints that turn dq and dk back as they store them
  bool unrope_attention() const { return rope_attention() || (dtype == EMI_F32 && hd() % 16 == 0 && hd() <= 128); }
  bool rope_projection() const { return rope_attention() && tiles(D); }
  bool swiglu_epilogue() const { return dtype == EMI_BF16 && T() >= 256; }
};

struct Carve {                                            // consecutive 256-byte aligned pieces of a buffer
  uint8_t* base;
  size_t at;
  void* take(size_t bytes) {
    void* p = base + at;
    at += (bytes + 255) / 256 * 256;
    return p;
  }
};
inline void* part(void* p, size_t bytes) { return static_cast<uint8_t*>(p) + bytes; }
inline const void* part(const void* p, size_t bytes) { return static_cast<const uint8_t*>(p) + bytes; }

struct Saved {                                            // of one layer
  void *xb1, *q, *k, *v, *att, *x1, *xb2, *h1, *h3, *g, *out;
  float* lse;
};
Saved carve_saved(void* base, const Dims& d, size_t* bytes = nullptr) {
  Carve c{static_cast<uint8_t*>(base), 0};
  const size_t td = (size_t)d.T() * d.D * d.elt(), th = (size_t)d.T() * d.H * d.elt();
  Saved s;
  s.xb1 = c.take(td);
  s.q = c.take(3 * td);                                   // side by side: q and k are rotated by one launch
  s.k = part(s.q, td);
  s.v = part(s.q, 2 * td);
  s.att = c.take(td);
  s.x1 = c.take(td);
  s.xb2 = c.take(td);
  s.h1 = c.take(th);
  s.h3 = c.take(th);
  s.g = c.take(th);
  s.out = c.take(td);
  s.lse = static_cast<float*>(c.take((size_t)d.B * d.heads * d.S * sizeof(float)));
  if (bytes != nullptr) *bytes = c.at;
  return s;
}

struct Cots {                                             // cotangents of one layer
  void *dq, *dk, *dv, *dx1, *dh1, *dh3, *dx;
};
Cots carve_cots(void* base, const Dims& d, size_t* bytes = nullptr) {
  Carve c{static_cast<uint8_t*>(base), 0};
  const size_t td = (size_t)d.T() * d.D * d.elt(), th = (size_t)d.T() * d.H * d.elt();
  Cots s;
  s.dq = c.take(3 * td);
  s.dk = part(s.dq, td);
  s.dv = part(s.dq, 2 * td);
  s.dx1 = c.take(td);
  s.dh1 = c.take(th);
  s.dh3 = c.take(th);
  s.dx = c.take(td);
  if (bytes != nullptr) *bytes = c.at;
  return s;
}

size_t most(std::initializer_list<size_t> v) {
  size_t m = 0;
  for (size_t x : v)
    if (x > m) m = x;
  return m;
}

size_t forward_scratch(const Dims& d) {
  const int64_t T = d.T();
  return most({emi_gemm_grouped_workspace_bytes(3, T, d.D, d.D, 0, 1, 0, d.dtype), emi_gemm_grouped_workspace_bytes(2, T, d.H, d.D, 0, 1, 0, d.dtype),
               emi_gemm_workspace_bytes(T, d.D, d.D, 0, 1, d.dtype), emi_gemm_workspace_bytes(T, d.H, d.D, 0, 1, d.dtype),
               emi_gemm_workspace_bytes(T, d.D, d.H, 0, 1, d.dtype)});
}

// dgamma's partial rows wait until the group is done and are summed by one launch
bool norms_wait(const Dims& d) { return emi::rmsnorm_one_pass(d.D); }
size_t norm_part_bytes(const Dims& d) { return (size_t)emi::rmsnorm_partial_rows(d.T(), d.D) * d.D * sizeof(float); }

struct ReverseScratch {
  void *dxb, *dg, *ws;
  size_t ws_bytes;
  float* parts;                                           // partial rows of dgamma, two adjoints a layer of the group
};
ReverseScratch carve_reverse(void* base, const Dims& d, int group, int transposed, size_t* bytes) {
  Carve c{static_cast<uint8_t*>(base), 0};
  const int64_t T = d.T();
  ReverseScratch s;
  s.dxb = c.take((size_t)T * d.D * d.elt());
  s.dg = c.take((size_t)T * d.H * d.elt());
  const int tb = transposed;
  int m4 = 4 * group, m2 = 2 * group, m1 = group;
  if (m4 > 48) m4 = 48;
  if (m2 > 48) m2 = 48;
  if (m1 > 48) m1 = 48;
  size_t need = most({emi_gemm_workspace_bytes(T, d.H, d.D, 0, tb, d.dtype), emi_gemm_workspace_bytes(T, d.D, d.D, 0, tb, d.dtype),
                      emi_gemm_grouped_workspace_bytes(2, T, d.D, d.H, 0, tb, 1, d.dtype),
                      emi_gemm_grouped_workspace_bytes(3, T, d.D, d.D, 0, tb, 1, d.dtype), emi_rmsnorm_bwd_workspace_bytes(T, d.D),
                      emi_attn_bwd_workspace_bytes(d.B, d.heads, d.S, d.hd())});
  for (int i = 1; i <= m4; i++) need = most({need, emi_gemm_grouped_workspace_bytes(i, d.D, d.D, T, 1, 0, 0, d.dtype)});
  for (int i = 1; i <= m2; i++) need = most({need, emi_gemm_grouped_workspace_bytes(i, d.H, d.D, T, 1, 0, 0, d.dtype)});
  for (int i = 1; i <= m1; i++) need = most({need, emi_gemm_grouped_workspace_bytes(i, d.D, d.H, T, 1, 0, 0, d.dtype)});
  s.ws_bytes = need;
  s.ws = c.take(need);
  s.parts = static_cast<float*>(c.take(norms_wait(d) ? 2 * (size_t)group * norm_part_bytes(d) : 0));
  if (bytes != nullptr) *bytes = c.at;
  return s;
}

#define EMI_TRY(call)            \
  do {                           \
    if (int rc__ = (call)) return rc__; \
  } while (0)

// y = rmsnorm(x) gamma, with x = a b^T + r by the product that comes before it.
int product_and_norm(emi_stream_t st, const void* a, const void* b, const void* r, void* x, const void* gamma, void* y, void* ws, size_t wsb,
                     int64_t K, const Dims& d) {
  int planes = 0;
  EMI_TRY(emi::gemm_run(static_cast<hipStream_t>(st), a, b, r, x, ws, wsb, d.T(), d.D, K, K, K, d.D, d.D, 0, 1, d.dtype,
                        emi::rmsnorm_one_pass(d.D) ? &planes : nullptr));
  if (planes > 0)
    return emi::launch_rmsnorm_fwd_planes(static_cast<hipStream_t>(st), static_cast<const float*>(ws), planes, r, gamma, x, y, d.T(), d.D, d.eps,
                                          d.dtype);
  return emi_rmsnorm_fwd(st, x, gamma, y, d.T(), d.D, d.eps, d.dtype);
}

// q, k, v from s.xb1, the normalised x.
int forward_heads(emi_stream_t st, const void* const* w, const float* table, const Saved& s, void* ws, size_t wsb, const Dims& d) {
  const int64_t T = d.T(), D = d.D;
  if (d.rope_projection()) {
    EMI_TRY(emi_gemm_rope(st, s.xb1, w[kQ], s.q, table, T, D, D, d.S, d.hd(), d.dtype));
    EMI_TRY(emi_gemm_rope(st, s.xb1, w[kK], s.k, table, T, D, D, d.S, d.hd(), d.dtype));
    EMI_TRY(emi_gemm_ws(st, s.xb1, w[kV], nullptr, s.v, ws, wsb, T, D, D, D, D, D, D, 0, 1, d.dtype));
  } else {
    emi::ProductTail t{emi::kTailRotated, {w[kQ], w[kK], w[kV]}, {s.q, s.k, s.v}, table, (int)d.S, (int)d.hd(), 2, 3, nullptr, nullptr, nullptr, {}};
    if (const int rc = emi::gemm_tail(static_cast<hipStream_t>(st), s.xb1, w[kQ], t, T, D, D, D, 1, d.dtype); rc > 0) return rc;
    else if (rc < 0) {
      const void *a[3] = {s.xb1, s.xb1, s.xb1}, *b[3] = {w[kQ], w[kK], w[kV]};
      void* c[3] = {s.q, s.k, s.v};
      EMI_TRY(emi_gemm_grouped(st, 3, a, b, nullptr, c, ws, wsb, T, D, D, D, D, D, D, 0, 1, 0, d.dtype));
      EMI_TRY(emi_rope(st, s.q, table, s.q, 2 * d.B, d.S, d.heads, d.hd(), 0, d.dtype));
    }
  }
  return EMI_OK;
}
int forward_attention(emi_stream_t st, const Saved& s, const Dims& d) {
  return emi_attn_fwd(st, s.q, s.k, s.v, s.att, s.lse, d.B, d.heads, d.S, d.hd(), d.S * d.D, d.hd(), d.D, d.scale, 1, d.dtype);
}

// h1, h3 and the SwiGLU from s.xb2, the normalised x1.
int forward_gated(emi_stream_t st, const void* const* w, const Saved& s, void* ws, size_t wsb, const Dims& d) {
  const int64_t T = d.T(), D = d.D, H = d.H;
  emi::ProductTail t{emi::kTailGated, {w[kW1], w[kW3], nullptr}, {s.h1, s.h3, s.g}, nullptr, 0, 0, 0, 0, nullptr, nullptr, nullptr, {}};
  if (const int rc = emi::gemm_tail(static_cast<hipStream_t>(st), s.xb2, w[kW1], t, T, H, D, D, 1, d.dtype); rc > 0) {
    return rc;
  } else if (rc == 0) {
  } else if (d.swiglu_epilogue()) {
    EMI_TRY(emi_gemm_ws(st, s.xb2, w[kW1], nullptr, s.h1, ws, wsb, T, H, D, D, D, H, H, 0, 1, d.dtype));
    EMI_TRY(emi_gemm_swiglu_fwd(st, s.xb2, w[kW3], s.h1, s.h3, s.g, T, H, D, d.dtype));
  } else {
    const void *a[2] = {s.xb2, s.xb2}, *b[2] = {w[kW1], w[kW3]};
    void* c[2] = {s.h1, s.h3};
    EMI_TRY(emi_gemm_grouped(st, 2, a, b, nullptr, c, ws, wsb, T, H, D, D, D, H, H, 0, 1, 0, d.dtype));
    EMI_TRY(emi_swiglu_fwd(st, s.h1, s.h3, s.g, T * H, d.dtype));
  }
  return EMI_OK;
}

// The layer's result; with the next layer's gamma its xb1 too.
int forward_result(emi_stream_t st, const void* const* w, const Saved& s, void* out, const void* next_gamma, void* next_xb, void* ws, size_t wsb,
                   const Dims& d) {
  if (next_xb != nullptr) return product_and_norm(st, s.g, w[kW2], s.x1, out, next_gamma, next_xb, ws, wsb, d.H, d);
  return emi_gemm_ws(st, s.g, w[kW2], s.x1, out, ws, wsb, d.T(), d.D, d.H, d.H, d.H, d.D, d.D, 0, 1, d.dtype);
}

// From s.xb1 on.
int forward_layer(emi_stream_t st, const void* const* w, const void* x, const float* table, const Saved& s, void* out, const void* next_gamma,
                  void* next_xb, void* ws, size_t wsb, const Dims& d) {
  EMI_TRY(forward_heads(st, w, table, s, ws, wsb, d));
  EMI_TRY(forward_attention(st, s, d));
  EMI_TRY(product_and_norm(st, s.att, w[kO], x, s.x1, w[kFfn], s.xb2, ws, wsb, d.D, d));
  EMI_TRY(forward_gated(st, w, s, ws, wsb, d));
  return forward_result(st, w, s, out, next_gamma, next_xb, ws, wsb, d);
}

// ---- forward mode: a layer's values and tangents ---------------------------------------------------------------

struct Tangents {                                         // of one layer
  void *xb, *q, *k, *v, *att, *x1, *h1, *h3, *g, *out;
};
// One set for all layers: a layer's result and the next one's xb1 go where its own x and xb1 have been read for the last time, the
// second norm's tangent where the first one's was, h1 and its tangent where q, k, v and att were.  The fewer bytes, the more of
// them the memory-side cache holds.
struct JvpScratch {
  Saved s;
  Tangents t;
  void* ws;
  size_t ws_bytes;
};
JvpScratch carve_jvp(void* base, const Dims& d, size_t* bytes = nullptr) {
  Carve c{static_cast<uint8_t*>(base), 0};
  const int64_t T = d.T();
  const size_t td = (size_t)T * d.D * d.elt(), th = (size_t)T * d.H * d.elt();
  const size_t heads = 4 * td > th ? 4 * td : th;
  JvpScratch s;
  s.s.xb1 = c.take(td);
  s.s.h1 = s.s.q = c.take(heads);
  s.s.k = part(s.s.q, td);
  s.s.v = part(s.s.q, 2 * td);
  s.s.att = part(s.s.q, 3 * td);
  s.s.x1 = c.take(td);
  s.s.xb2 = c.take(td);
  s.s.h3 = c.take(th);
  s.s.g = c.take(th);
  s.s.out = c.take(td);
  s.s.lse = static_cast<float*>(c.take((size_t)d.B * d.heads * d.S * sizeof(float)));
  s.t.xb = c.take(td);
  s.t.h1 = s.t.q = c.take(heads);
  s.t.k = part(s.t.q, td);
  s.t.v = part(s.t.q, 2 * td);
  s.t.att = part(s.t.q, 3 * td);
  s.t.x1 = c.take(td);
  s.t.h3 = c.take(th);
  s.t.g = c.take(th);
  s.t.out = c.take(td);
  s.ws_bytes = most({forward_scratch(d), emi_gemm_grouped_workspace_bytes(2, T, d.D, d.D, 0, 1, 1, d.dtype),
                     emi_gemm_grouped_workspace_bytes(2, T, d.H, d.D, 0, 1, 1, d.dtype), emi_gemm_grouped_workspace_bytes(2, T, d.D, d.H, 0, 1, 1, d.dtype)});
  s.ws = c.take(s.ws_bytes);
  if (bytes != nullptr) *bytes = c.at;
  return s;
}

// Estimates for one result of tangent_product: its two products one by one, and as one launch that sums them.
struct TangentPlan {
  double two, sum;
  int64_t splits;
};
TangentPlan tangent_plan(int64_t N, int64_t K, const JvpScratch& k, const Dims& d) {
  const int64_t T = d.T(), held = emi::splits_held(k.ws, k.ws_bytes, T, N), most = emi::sum_splits(T, N, held);
  if (d.dtype == EMI_F32) return {2 * emi::f32_plan(T, N, K, 1, 0, 0, held).us + 1.0, emi::f32_plan(T, N, K, 2, 1, 0, most).us, most};
  // (long sums that fill the chip run a tenth longer than estimated: two of 1000 x 4096 x 4096 84 us, one by one 80)
  return {2 * emi::bf16_plan(T, N, K, 1, 0, 1, held).us + 1.0, emi::bf16_plan(T, N, K, 2, 1, 1, most).us * (most > 1 ? 1.0 : 1.1), most};
}

// ty = tx w^T + x tw^T [+ r].  As two products in the operators' order: w, which the value's own product has just read, is still in
// the memory-side cache, and the sum is added to while it is.  bf16, dim 4096, us a layer, the other way round and the results
// that share x in turn | this (operator by operator): 1500 tokens 2389 | 2374 (2411), 2000 2760 | 2752 (2756).
int tangent_product(emi_stream_t st, const void* tx, const void* x, const void* w, const void* tw, const void* r, void* ty, int64_t N, int64_t K,
                    const JvpScratch& k, const Dims& d) {
  const int64_t T = d.T();
  const TangentPlan p = tangent_plan(N, K, k, d);
  if (p.two < p.sum) {
    EMI_TRY(emi_gemm_ws(st, tx, w, r, ty, k.ws, k.ws_bytes, T, N, K, K, K, N, N, 0, 1, d.dtype));
    return emi_gemm_ws(st, x, tw, ty, ty, k.ws, k.ws_bytes, T, N, K, K, K, N, N, 0, 1, d.dtype);
  }
  const void *a[2] = {tx, x}, *b[2] = {w, tw}, *res[1] = {r};
  void* out[1] = {ty};
  return emi_gemm_grouped(st, 2, a, b, r != nullptr ? res : nullptr, out, p.splits > 1 ? k.ws : nullptr, p.splits > 1 ? k.ws_bytes : 0, T, N, K, K, K, N, N,
                          0, 1, 1, d.dtype);
}

// Several results of tangent_product that share x and tx; the first `rotated` turned.  One launch where that is faster, or the
// products with every w as one group and those with every tw, which add to them, as another (bf16: the 256-tiles of three
// results fill the chip where one's do not, 1000 x 4096 x 4096 180 us, result by result 241; where one's do, a group would
// run one by one, every sum out of the cache before it is added to: 2000 x 11008 x 4096 194 us a second product, 188 behind the first).
int tangent_products(emi_stream_t st, const void* tx, const void* x, std::initializer_list<int> which, const void* const* w, const void* const* tw,
                     std::initializer_list<void*> out, int rotated, const float* table, int64_t N, const JvpScratch& k, const Dims& d) {
  emi::ProductTail t{emi::kTailRotated, {}, {}, rotated ? table : nullptr, (int)d.S, (int)d.hd(), rotated, 0, nullptr, nullptr, x, {}};
  for (int i : which) {
    t.B[t.count] = w[i];
    t.B1[t.count] = tw[i];
    t.C[t.count] = out.begin()[t.count];
    t.count++;
  }
  const int rc = emi::gemm_tail(static_cast<hipStream_t>(st), tx, t.B[0], t, d.T(), N, d.D, d.D, 1, d.dtype);
  if (rc >= 0) return rc;
  const TangentPlan p = tangent_plan(N, d.D, k, d);
  const double group = d.dtype == EMI_F32 ? emi::f32_plan(d.T(), N, d.D, t.count, 0, 0, 1).us : emi::bf16_plan(d.T(), N, d.D, t.count, 0, 1, 1).us;
  const bool one_launch = d.dtype == EMI_F32 || emi::bf16_one_launch(d.T(), N);
  if (one_launch && 2 * group + 1.0 < t.count * ((p.two < p.sum ? p.two : p.sum) + 1.0)) {
    const void *xs[3] = {x, x, x}, *txs[3] = {tx, tx, tx};
    EMI_TRY(emi_gemm_grouped(st, t.count, txs, t.B, nullptr, t.C, k.ws, k.ws_bytes, d.T(), N, d.D, d.D, d.D, N, N, 0, 1, 0, d.dtype));
    EMI_TRY(emi_gemm_grouped(st, t.count, xs, t.B1, t.C, t.C, k.ws, k.ws_bytes, d.T(), N, d.D, d.D, d.D, N, N, 0, 1, 0, d.dtype));
  } else {
    for (int i = 0; i < t.count; i++) EMI_TRY(tangent_product(st, tx, x, t.B[i], t.B1[i], nullptr, t.C[i], N, d.D, k, d));
  }
  return rotated ? emi_rope(st, t.C[0], table, t.C[0], rotated * d.B, d.S, d.heads, d.hd(), 0, d.dtype) : EMI_OK;      // (side by side)
}

// A layer from s.xb1 on and its tangents; tx: the tangent of its input x.  Each tangent behind the values it is of: they share
// weights and activations, which the memory-side cache keeps from one to the other.  us, all values first and a set of buffers for
// odd and one for even layers | this, bf16: 4096 tokens at dim 2048 1755 | 1705, 16384 6214 | 6100, 16384 at dim 1024 2873 | 2835,
// 5784 at dim 768 843 | 841.
int tangent_layer(emi_stream_t st, const void* const* w, const void* const* tw, const void* x, const void* tx, const float* table,
                  const JvpScratch& k, void* out, void* tout, const void* next_gamma, void* next_xb, const Dims& d) {
  const Saved& s = k.s;
  const Tangents& t = k.t;
  const int64_t T = d.T(), D = d.D, H = d.H;
  EMI_TRY(emi_rmsnorm_jvp(st, x, w[kAtt], tx, tw[kAtt], t.xb, T, D, d.eps, d.dtype));
  EMI_TRY(forward_heads(st, w, table, s, k.ws, k.ws_bytes, d));
  EMI_TRY(tangent_products(st, t.xb, s.xb1, {kQ, kK, kV}, w, tw, {t.q, t.k, t.v}, 2, table, D, k, d));
  EMI_TRY(forward_attention(st, s, d));
  EMI_TRY(emi_attn_jvp(st, s.q, s.k, s.v, s.lse, t.q, t.k, t.v, t.att, d.B, d.heads, d.S, d.hd(), d.S * D, d.hd(), D, d.scale, 1, d.dtype));
  EMI_TRY(product_and_norm(st, s.att, w[kO], x, s.x1, w[kFfn], s.xb2, k.ws, k.ws_bytes, D, d));
  EMI_TRY(tangent_product(st, t.att, s.att, w[kO], tw[kO], tx, t.x1, D, D, k, d));
  EMI_TRY(emi_rmsnorm_jvp(st, s.x1, w[kFfn], t.x1, tw[kFfn], t.xb, T, D, d.eps, d.dtype));
  EMI_TRY(forward_gated(st, w, s, k.ws, k.ws_bytes, d));
  EMI_TRY(tangent_products(st, t.xb, s.xb2, {kW1, kW3}, w, tw, {t.h1, t.h3}, 0, nullptr, H, k, d));
  EMI_TRY(emi_swiglu_jvp(st, s.h1, s.h3, t.h1, t.h3, t.g, T * H, d.dtype));
  EMI_TRY(forward_result(st, w, s, out, next_gamma, next_xb, k.ws, k.ws_bytes, d));
  return tangent_product(st, t.g, s.g, w[kW2], tw[kW2], t.x1, tout, D, H, k, d);
}

// dW = dY^T X of one shape, waiting to run as one launch.
struct Pending {
  const void *a[48], *b[48];
  void* c[48];
  int n = 0;
};
int flush(emi_stream_t st, Pending& p, int64_t M, int64_t N, int64_t T, const ReverseScratch& r, int dtype) {
  if (p.n == 0) return EMI_OK;
  const int n = p.n;
  p.n = 0;
  if (n == 1) return emi_gemm_ws(st, p.a[0], p.b[0], nullptr, p.c[0], r.ws, r.ws_bytes, M, N, T, M, N, N, N, 1, 0, dtype);
  return emi_gemm_grouped(st, n, p.a, p.b, nullptr, p.c, r.ws, r.ws_bytes, M, N, T, M, N, N, N, 1, 0, 0, dtype);
}
int wait(emi_stream_t st, Pending& p, const void* dy, const void* x, void* dw, int64_t M, int64_t N, int64_t T, const ReverseScratch& r,
         int dtype) {
  if (p.n == 48) EMI_TRY(flush(st, p, M, N, T, r, dtype));
  p.a[p.n] = dy;
  p.b[p.n] = x;
  p.c[p.n++] = dw;
  return EMI_OK;
}

// RMSNorm adjoints whose column sums wait.
struct Norms {
  emi::Colsums c;
  int n = 0;
};
int flush(emi_stream_t st, Norms& p, const Dims& d) {
  const int n = p.n;
  p.n = 0;
  return emi::launch_colsums(static_cast<hipStream_t>(st), p.c, n, emi::rmsnorm_partial_rows(d.T(), d.D), d.D, d.dtype);
}
// dy in `dy`, or in `planes` planes of the workspace.
int norm_adjoint(emi_stream_t st, Norms& p, const void* x, const void* gamma, const void* dy, int planes, const void* dx_add, void* dx,
                 void* dgamma, const ReverseScratch& r, const Dims& d) {
  if (!norms_wait(d)) return emi_rmsnorm_bwd(st, x, gamma, dy, dx_add, dx, dgamma, r.ws, r.ws_bytes, d.T(), d.D, d.eps, d.dtype);
  if (p.n == emi::kMaxColsums) EMI_TRY(flush(st, p, d));
  float* part_rows = reinterpret_cast<float*>(reinterpret_cast<uint8_t*>(r.parts) + p.n * norm_part_bytes(d));
  p.c.part[p.n] = part_rows;
  p.c.out[p.n++] = dgamma;
  return emi::launch_rmsnorm_bwd_rows(static_cast<hipStream_t>(st), x, gamma, planes > 0 ? r.ws : dy, planes, dx_add, dx, part_rows, d.T(), d.D, d.eps, d.dtype);
}

int check_layers(const char* name, const Dims& d, const void* const* w, std::initializer_list<const void*> ptrs) {
  if (!d.ok())
    return emi_fail(EMI_INVALID_ARGUMENT, "%s: unsupported shape (layers=%lld batch=%lld seq=%lld dim=%lld hidden=%lld heads=%lld dtype=%d)", name,
                    (long long)d.L, (long long)d.B, (long long)d.S, (long long)d.D, (long long)d.H, (long long)d.heads, d.dtype);
  if (w == nullptr) return emi_fail(EMI_INVALID_ARGUMENT, "%s: null weight table", name);
  for (int i = 0; i < kWeights; i++)
    if (w[i] == nullptr) return emi_fail(EMI_INVALID_ARGUMENT, "%s: weight %d is null", name, i);
  for (const void* p : ptrs)
    if (p == nullptr) return emi_fail(EMI_INVALID_ARGUMENT, "%s: null buffer", name);
  return EMI_OK;
}

size_t weight_elements(int i, const Dims& d) {            // of one layer
  switch (i) {
    case kAtt: case kFfn: return (size_t)d.D;
    case kW1: case kW2: case kW3: return (size_t)d.D * d.H;
    default: return (size_t)d.D * d.D;
  }
}

}  // namespace

extern "C" size_t emi_llama_layers_saved_bytes(int64_t batch, int64_t seq, int64_t dim, int64_t hidden, int64_t heads, int dtype) {
  const Dims d{1, batch, seq, dim, hidden, heads, 0.f, 0.f, dtype};
  if (!d.ok()) return 0;
  size_t n = 0;
  carve_saved(nullptr, d, &n);
  return n;
}

extern "C" size_t emi_llama_layers_fwd_workspace_bytes(int64_t batch, int64_t seq, int64_t dim, int64_t hidden, int64_t heads, int dtype) {
  const Dims d{1, batch, seq, dim, hidden, heads, 0.f, 0.f, dtype};
  return d.ok() ? forward_scratch(d) : 0;
}

extern "C" size_t emi_llama_layers_cotangent_bytes(int64_t batch, int64_t seq, int64_t dim, int64_t hidden, int64_t heads, int dtype) {
  const Dims d{1, batch, seq, dim, hidden, heads, 0.f, 0.f, dtype};
  if (!d.ok()) return 0;
  size_t n = 0;
  carve_cots(nullptr, d, &n);
  return n;
}

extern "C" size_t emi_llama_layers_bwd_workspace_bytes(int64_t batch, int64_t seq, int64_t dim, int64_t hidden, int64_t heads, int group,
                                                       int transposed, int dtype) {
  const Dims d{1, batch, seq, dim, hidden, heads, 0.f, 0.f, dtype};
  if (!d.ok() || group < 1) return 0;
  size_t n = 0;
  carve_reverse(nullptr, d, group, transposed, &n);
  return n;
}

extern "C" int emi_llama_layers_fwd(emi_stream_t stream, const void* const* weights, const void* x, const float* rope_table, void* y,
                                    void* const* saved, int keep, void* workspace, size_t workspace_bytes, int64_t layers, int64_t batch,
                                    int64_t seq, int64_t dim, int64_t hidden, int64_t heads, float eps, float scale, int dtype) {
  const Dims d{layers, batch, seq, dim, hidden, heads, eps, scale, dtype};
  if (int rc = check_layers("emi_llama_layers_fwd", d, weights, {x, rope_table, y, saved})) return rc;
  const size_t need = forward_scratch(d);
  if (need && (workspace == nullptr || workspace_bytes < need))
    return emi_fail(EMI_INVALID_ARGUMENT, "emi_llama_layers_fwd: workspace of %zu bytes needed, got %zu", need, workspace_bytes);
  for (int64_t l = 0; l < layers; l++) {
    const void* w[kWeights];
    for (int i = 0; i < kWeights; i++) w[i] = part(weights[i], weight_elements(i, d) * (size_t)l * d.elt());
    void* buffer = saved[keep ? l : 0];
    if (buffer == nullptr) return emi_fail(EMI_INVALID_ARGUMENT, "emi_llama_layers_fwd: null buffer for layer %lld", (long long)l);
    const Saved s = carve_saved(buffer, d);
    void* out = l + 1 < layers ? s.out : y;
    void* next = l + 1 < layers ? saved[keep ? l + 1 : 0] : nullptr;
    if (l + 1 < layers && next == nullptr)
      return emi_fail(EMI_INVALID_ARGUMENT, "emi_llama_layers_fwd: null buffer for layer %lld", (long long)(l + 1));
    if (l == 0) EMI_TRY(emi_rmsnorm_fwd(stream, x, w[kAtt], s.xb1, d.T(), dim, eps, dtype));
    EMI_TRY(forward_layer(stream, w, x, rope_table, s, out, part(weights[kAtt], (size_t)dim * (size_t)(l + 1) * d.elt()),
                          next != nullptr ? carve_saved(next, d).xb1 : nullptr, workspace, workspace_bytes, d));
    x = out;
  }
  return EMI_OK;
}

extern "C" int emi_llama_layers_bwd(emi_stream_t stream, const void* const* weights, void* const* transposed, const void* x,
                                    const float* rope_table, void* const* saved, const void* dy, const void* dx_add, void* dx,
                                    void* const* grads, void* const* cotangents, int group, void* workspace, size_t workspace_bytes,
                                    int64_t layers, int64_t batch, int64_t seq, int64_t dim, int64_t hidden, int64_t heads, float eps,
                                    float scale, int dtype) {
  const Dims d{layers, batch, seq, dim, hidden, heads, eps, scale, dtype};
  if (int rc = check_layers("emi_llama_layers_bwd", d, weights, {x, rope_table, saved, dy, dx, grads, cotangents, workspace})) return rc;
  if (group < 1) return emi_fail(EMI_INVALID_ARGUMENT, "emi_llama_layers_bwd: group %d", group);
  for (int i = 0; i < kWeights; i++)
    if (grads[i] == nullptr) return emi_fail(EMI_INVALID_ARGUMENT, "emi_llama_layers_bwd: gradient %d is null", i);
  size_t need = 0;
  const ReverseScratch r = carve_reverse(workspace, d, group, transposed != nullptr, &need);
  if (workspace_bytes < need)
    return emi_fail(EMI_INVALID_ARGUMENT, "emi_llama_layers_bwd: workspace of %zu bytes needed, got %zu", need, workspace_bytes);
  const int64_t T = d.T(), D = d.D, H = d.H;
  const int tb = transposed != nullptr;                   // dX = dY . W as NT on W^T, or NN on W as stored
  if (tb)
    for (int i : {kQ, kK, kV, kO, kW1, kW2, kW3}) {       // every layer's transpose by one launch per stack
      if (transposed[i] == nullptr) return emi_fail(EMI_INVALID_ARGUMENT, "emi_llama_layers_bwd: no room for transpose %d", i);
      const int64_t rows = i == kW1 || i == kW3 ? H : D, cols = i == kW2 ? H : D;
      const int64_t out[3] = {layers, cols, rows}, ss[3] = {rows * cols, 1, cols}, ds[3] = {rows * cols, rows, 1};
      EMI_TRY(layers == 1 ? emi_transpose(stream, weights[i], transposed[i], rows, cols, dtype)
                          : emi_strided_copy(stream, weights[i], transposed[i], 3, out, ss, 0, ds, 0, (int)d.elt()));
    }
  Pending sq, up, down;                                   // [D, D], [H, D], [D, H]
  Norms norms;
  int planes = 0;                                         // of the product that the next RMSNorm adjoint reads
  int* const leave = norms_wait(d) ? &planes : nullptr;
  const int64_t hd = d.hd();
  for (int64_t l = layers - 1; l >= 0; l--) {
    const void *w[kWeights], *b[kWeights];
    void* g[kWeights];
    for (int i = 0; i < kWeights; i++) {
      const size_t off = weight_elements(i, d) * (size_t)l * d.elt();
      w[i] = part(weights[i], off);
      b[i] = tb && transposed[i] != nullptr ? part(static_cast<const void*>(transposed[i]), off) : w[i];
      g[i] = part(grads[i], off);
    }
    const Saved s = carve_saved(saved[l], d);
    const int64_t done = layers - 1 - l;
    const Cots c = carve_cots(cotangents[done % group], d);
    const void* x_l = l == 0 ? x : carve_saved(saved[l - 1], d).out;
    EMI_TRY(wait(stream, down, dy, s.g, g[kW2], D, H, T, r, dtype));
    // the group's last layer writes its dx where the dy of the group's first one lies (the last slot's dx, of the group before)
    const bool ends_group = (done + 1) % group == 0 || l == 0;
    if (ends_group) EMI_TRY(flush(stream, down, D, H, T, r, dtype));
    emi::ProductTail t{emi::kTailAdjoint, {}, {c.dh1, c.dh3, nullptr}, nullptr, 0, 0, 0, 0, s.h1, s.h3, nullptr, {}};
    if (const int rc = emi::gemm_tail(static_cast<hipStream_t>(stream), dy, b[kW2], t, T, H, D, tb ? D : H, tb, dtype); rc > 0) {
      return rc;
    } else if (rc == 0) {
    } else if (tb && d.swiglu_epilogue()) {
      EMI_TRY(emi_gemm_swiglu_bwd(stream, dy, b[kW2], s.h1, s.h3, c.dh1, c.dh3, r.dg, (size_t)T * H * d.elt(), T, H, D, dtype));
    } else {
      EMI_TRY(emi_gemm_ws(stream, dy, b[kW2], nullptr, r.dg, r.ws, r.ws_bytes, T, H, D, D, tb ? D : H, H, H, 0, tb, dtype));
      EMI_TRY(emi_swiglu_bwd(stream, s.h1, s.h3, r.dg, c.dh1, c.dh3, T * H, dtype));
    }
    {
      const void *a2[2] = {c.dh1, c.dh3}, *b2[2] = {b[kW1], b[kW3]};
      void* out[1] = {r.dxb};
      EMI_TRY(emi::gemm_grouped_run(static_cast<hipStream_t>(stream), 2, a2, b2, nullptr, out, r.ws, r.ws_bytes, T, D, H, H, tb ? H : D, D, D, 0,
                                    tb, 1, dtype, leave));
    }
    EMI_TRY(norm_adjoint(stream, norms, s.x1, w[kFfn], r.dxb, planes, dy, c.dx1, g[kFfn], r, d));
    EMI_TRY(emi_gemm_ws(stream, c.dx1, b[kO], nullptr, r.dxb, r.ws, r.ws_bytes, T, D, D, D, D, D, D, 0, tb, dtype));
    if (d.unrope_attention()) {
      EMI_TRY(emi_attn_bwd_rope(stream, s.q, s.k, s.v, s.att, s.lse, r.dxb, c.dq, c.dk, c.dv, rope_table, r.ws, r.ws_bytes, d.B, d.heads, d.S, hd,
                                d.S * D, hd, D, d.scale, 1, dtype));
    } else {
      EMI_TRY(emi_attn_bwd(stream, s.q, s.k, s.v, s.att, s.lse, r.dxb, c.dq, c.dk, c.dv, r.ws, r.ws_bytes, d.B, d.heads, d.S, hd, d.S * D, hd, D,
                           d.scale, 1, dtype));
      EMI_TRY(emi_rope(stream, c.dq, rope_table, c.dq, 2 * d.B, d.S, d.heads, hd, 1, dtype));
    }
    {
      const void *a3[3] = {c.dq, c.dk, c.dv}, *b3[3] = {b[kQ], b[kK], b[kV]};
      void* out[1] = {r.dxb};
      EMI_TRY(emi::gemm_grouped_run(static_cast<hipStream_t>(stream), 3, a3, b3, nullptr, out, r.ws, r.ws_bytes, T, D, D, D, D, D, D, 0, tb, 1, dtype,
                                    leave));
    }
    // the first layer's cotangent leaves; a caller's accumulated one is added by its own launch
    void* dx_l = l == 0 ? dx : c.dx;
    EMI_TRY(norm_adjoint(stream, norms, x_l, w[kAtt], r.dxb, planes, c.dx1, dx_l, g[kAtt], r, d));
    if (l == 0 && dx_add != nullptr) EMI_TRY(emi_add(stream, dx, dx_add, dx, T * D, dtype));
    EMI_TRY(wait(stream, sq, c.dq, s.xb1, g[kQ], D, D, T, r, dtype));
    EMI_TRY(wait(stream, sq, c.dk, s.xb1, g[kK], D, D, T, r, dtype));
    EMI_TRY(wait(stream, sq, c.dv, s.xb1, g[kV], D, D, T, r, dtype));
    EMI_TRY(wait(stream, sq, c.dx1, s.att, g[kO], D, D, T, r, dtype));
    EMI_TRY(wait(stream, up, c.dh1, s.xb2, g[kW1], H, D, T, r, dtype));
    EMI_TRY(wait(stream, up, c.dh3, s.xb2, g[kW3], H, D, T, r, dtype));
    if (ends_group) {
      EMI_TRY(flush(stream, sq, D, D, T, r, dtype));
      EMI_TRY(flush(stream, up, H, D, T, r, dtype));
      EMI_TRY(flush(stream, norms, d));
    }
    dy = dx_l;
  }
  return EMI_OK;
}

extern "C" size_t emi_llama_layers_jvp_workspace_bytes(int64_t batch, int64_t seq, int64_t dim, int64_t hidden, int64_t heads, int dtype) {
  const Dims d{1, batch, seq, dim, hidden, heads, 0.f, 0.f, dtype};
  if (!d.ok()) return 0;
  size_t n = 0;
  carve_jvp(nullptr, d, &n);
  return n;
}

extern "C" int emi_llama_layers_jvp(emi_stream_t stream, const void* const* weights, const void* const* tangents, const void* x, const void* tx,
                                    const float* rope_table, void* y, void* ty, void* workspace, size_t workspace_bytes, int64_t layers,
                                    int64_t batch, int64_t seq, int64_t dim, int64_t hidden, int64_t heads, float eps, float scale, int dtype) {
  const Dims d{layers, batch, seq, dim, hidden, heads, eps, scale, dtype};
  if (int rc = check_layers("emi_llama_layers_jvp", d, weights, {x, tx, rope_table, y, ty, workspace, tangents})) return rc;
  for (int i = 0; i < kWeights; i++)
    if (tangents[i] == nullptr) return emi_fail(EMI_INVALID_ARGUMENT, "emi_llama_layers_jvp: tangent %d is null", i);
  size_t need = 0;
  const JvpScratch k = carve_jvp(workspace, d, &need);
  if (workspace_bytes < need)
    return emi_fail(EMI_INVALID_ARGUMENT, "emi_llama_layers_jvp: workspace of %zu bytes needed, got %zu", need, workspace_bytes);
  for (int64_t l = 0; l < layers; l++) {
    const void *w[kWeights], *tw[kWeights];
    for (int i = 0; i < kWeights; i++) {
      const size_t off = weight_elements(i, d) * (size_t)l * d.elt();
      w[i] = part(weights[i], off);
      tw[i] = part(tangents[i], off);
    }
    const bool last = l + 1 == layers;
    if (l == 0) EMI_TRY(emi_rmsnorm_fwd(stream, x, w[kAtt], k.s.xb1, d.T(), dim, eps, dtype));
    void *out = last ? y : k.s.out, *tout = last ? ty : k.t.out;
    EMI_TRY(tangent_layer(stream, w, tw, x, tx, rope_table, k, out, tout, part(w[kAtt], last ? 0 : (size_t)dim * d.elt()), last ? nullptr : k.s.xb1, d));
    x = out;
    tx = tout;
  }
  return EMI_OK;
}
