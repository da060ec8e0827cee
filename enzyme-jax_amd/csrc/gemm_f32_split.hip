// fp32 products on the bf16 matrix cores.
//
//   C[M,N] = op(A) . op(B) [+ R]      fp32 in, fp32 out, errors no larger than those of the fp32 instructions
//
// A bf16 matrix instruction multiplies sixteen times as fast as an fp32 one.  An fp32 number is the sum of three bf16
// numbers, exactly: h = bf16(x), m = bf16(x - h), l = x - h - m (8 + 8 + 8 bits, the differences exact).  That holds from 2^-102
// on; a tile whose operands hold a smaller number (but 0) is multiplied in fp32 as it is, so that neither a row of small numbers
// nor a single one loses bits to its neighbours (rows of 1e-36 beside rows of N(0, 1): 1.4e-7; 2.7e-5 without that).  Of the nine
// products of two such sums hh, hm, mh, mm, hl, lh are taken; the other three are below 2^-25 of the whole.  Products of
// bf16 are exact and summed in fp32: hh in sums of their own, so that what the small ones round off is 2^-8 smaller, and
// both end in `total` every PF stages (64 or 96 k), which keeps the chains short.  Relative error against float64, this | the
// fp32 instructions with chains of 32: 2000 x 768 x 768 0.8e-7 | 1.3e-7, 4096^3 1.3e-7 | 2.3e-7, 256 x 288 x 32000 1.3e-7 | 1.9e-7.
// What bounds it: 6 products at the rate that random bf16 numbers leave the clock at (1.7 GHz: 300 TFLOP/s), and on a CU the
// issue of the split beside the matrix instructions, 5.5 instructions a number and 1.5 to 2 that test it, of which a wavefront issues
// one in 7.7 cycles.
// Measured, us, 64- and 128-tiles of the fp32 instructions | this: 2000 x 768 x 768 32.5 | 26.1; 2000 x 2048 x 768 59 | 41;
// 2048 x 768 x 2000 (TN, four) 223 | 170; 777 x 4096 x 4096 232 | 162; 4096^3 1008 | 730 (188 TFLOP/s).
// Wavefronts that only split beside others that only multiply, eight wavefronts a block instead of sixteen, fragments read a
// k-step ahead: all the same 1.03 us a stage of a 128 x 128 block, or slower.
#include <type_traits>

#include "emi_device.h"
#include "gemm_f32.h"

namespace emi {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16_t;
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
#define EMI_LDS __attribute__((address_space(3)))
constexpr uint32_t kOob = 0x80000000u;   // beyond any buffer's num_records: loads return 0
constexpr int kDenormal = 1 << 4 | 1 << 7;   // of v_cmp_class: negative, positive

// N numbers; h, m, l: two numbers in a word.  Step by step over all of them: an instruction that needs the result of the
// one before it waits for it.  rest: what is left for l.
template <int N>
__device__ __forceinline__ void split(const float (&x)[N], uint32_t (&h)[N / 2], uint32_t (&m)[N / 2], uint32_t (&l)[N / 2], float (&r)[N]) {
  float t[N];
  auto round = [&](uint32_t (&to)[N / 2], const float (&v)[N]) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < N / 2; q++) to[q] = pack_bf16x2(v[2 * q], v[2 * q + 1]);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto rest = [&](const uint32_t (&of)[N / 2], const float (&v)[N]) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < N; q++) t[q] = __uint_as_float(q & 1 ? of[q / 2] & 0xffff0000u : of[q / 2] << 16);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < N; q++) r[q] = v[q] - t[q];
    __builtin_amdgcn_sched_barrier(0);
  };
  round(h, x);
  rest(h, x);
  round(m, r);
  rest(m, r);
  round(l, r);
}

// One operand of a block: ROWS rows (of A: rows of C; of B: columns of C) by 32 of the contraction per stage, loaded
// into registers, split, and laid into the LDS as three planes of 16-byte pieces: [kp][slot], piece kp of a row holding the
// eight k  4 kp .. + 3 and 16 + 4 kp .. + 3, in that order.  A thread takes half a piece (1024 threads for 128 rows, 512 for 64)
// or a whole one (512 for 128), so that eight or four lanes read 128 or 64 consecutive bytes of a k-contiguous row.  slot(row) and the 32 bytes
// between the kp's spread the lanes of one pass of an LDS write over all banks.
template <int ROWS, int THREADS, int PF, bool KM> struct SplitOperand {
  static constexpr int KP = ROWS * 16 + 32, PLANE = 4 * KP, BYTES = 3 * PLANE;
  static constexpr int E = ROWS * 32 / THREADS;                      // numbers per thread and stage
  static_assert(E == 4 || E == 8, "a piece or half of one");
  static __device__ __forceinline__ int slot(int r) { return r ^ ((r >> 4) & 1); }
  static __device__ __forceinline__ int k_of(int e) { return e < 4 ? e : e + 12; }

  uint32_t voff, at;                                              // of the first number in memory, of the piece in the LDS
  int k0;                                                         // the first k
  float x[PF + 2][E];                                             // the stages in flight; two more to begin with
  // What has been split may have held a number that is not the sum of its parts: bf16 holds what is left for l, eight bits, unless
  // that is a denormal fp32 number, and from 2^-102 on it is 0 or at least 2^-126.  The class of what is left takes an
  // instruction of the vector and one of the scalar unit a number, the least number but 0 one and a half of the vector
  // unit; the second are fewer for a wavefront that is alone on its SIMD, the first hide among four.  us, neither | class |
  // least: 2000 x 768 x 768 (128 x 64) 26.3 | 28.9 | 26.6, 1000 x 768 x 768 (64 x 64) 18.1 | 19.1 | 18.7, 777 x 4096 x 4096
  // (128 x 128) 169 | 170 | 172, 2048^3 97.8 | 98.2 | 99.8.
  static constexpr bool BY_CLASS = THREADS == 1024;
  uint64_t lost;                                                  // lanes
  uint32_t least;                                                 // bits << 1, less one
  __device__ __forceinline__ bool inexact() const { return BY_CLASS ? lost != 0 : least < (25u << 24) - 1; }
  __device__ __forceinline__ void init(int rows_left, int ld) {
    const int tid = threadIdx.x;
    const int row = KM ? tid % ROWS : tid / (32 / E), q = KM ? tid / ROWS : tid % (32 / E);
    k0 = 4 * q;                                                   // E == 4: quad q of the 32 k; E == 8: quads q and q + 4
    lost = 0;
    least = 0xffffffffu;
    voff = row < rows_left ? (uint32_t)(KM ? k0 * ld + row : row * ld + k0) * 4u : kOob;
    at = (uint32_t)((q & 3) * KP + slot(row) * 16 + (q >> 2) * 8);
  }
  // corner: the operand at the block's first row and the stage's first k, of which `left` are left to contract
  __device__ __forceinline__ void load(int f, const float* corner, int rows, int ld, int left) {
    const uint32_t bytes = left <= 0 ? 0u : (uint32_t)(KM ? ((left < 32 ? left : 32) - 1) * ld + rows : (rows - 1) * ld + left) * 4u;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(corner), 0, bytes, 0x00020000);
    if constexpr (KM) {
#pragma unroll
      for (int e = 0; e < E; e++)                                  // (kOob stays beyond num_records)
        x[f][e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc, voff + (uint32_t)(k_of(e) * ld) * 4u, 0, 0));
    } else {
#pragma unroll
      for (int e = 0; e < E; e += 4) {
        uint32_t at = voff + 4u * k_of(e);
        if (left < 32) at = k0 + k_of(e) < left ? at : kOob;
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(rsrc, at, 0, 0);
#pragma unroll
        for (int c = 0; c < 4; c++) x[f][e + c] = __uint_as_float(v[c]);
      }
    }
  }
  __device__ __forceinline__ void store(int f, EMI_LDS uint8_t* lds) {
    uint32_t h[E / 2], m[E / 2], l[E / 2];
    float rest[E];
    split<E>(x[f], h, m, l, rest);
    if constexpr (BY_CLASS) {
      bool any = false;
#pragma unroll
      for (int q = 0; q < E; q++) any = any | __builtin_amdgcn_classf(rest[q], kDenormal);
      lost |= __builtin_amdgcn_ballot_w64(any);
    } else {
#pragma unroll
      for (int q = 0; q < E; q += 2)
        least = min(min(least, (__float_as_uint(x[f][q]) << 1) - 1), (__float_as_uint(x[f][q + 1]) << 1) - 1);      // 0 wraps round
    }
    put(lds + at, h);
    put(lds + at + PLANE, m);
    put(lds + at + 2 * PLANE, l);
  }
  static __device__ __forceinline__ void put(EMI_LDS uint8_t* to, const uint32_t (&v)[E / 2]) {
    if constexpr (E == 8)
      *reinterpret_cast<EMI_LDS u32x4_t*>(to) = u32x4_t{v[0], v[1], v[2], v[3]};
    else
      *reinterpret_cast<EMI_LDS u32x2_t*>(to) = u32x2_t{v[0], v[1]};
  }
  // The numbers as they are, for the tiles that are multiplied in fp32: [quad][slot] in pieces of four k.
  __device__ __forceinline__ void store_f32(int f, EMI_LDS uint8_t* lds) {
    EMI_LDS uint8_t* to = lds + (k0 >> 2) * KP + slot(KM ? threadIdx.x % ROWS : threadIdx.x / (32 / E)) * 16;
#pragma unroll
    for (int e = 0; e < E; e += 4)
      *reinterpret_cast<EMI_LDS f32x4_t*>(to + e * KP) = f32x4_t{x[f][e], x[f][e + 1], x[f][e + 2], x[f][e + 3]};      // quads q, q + 4
  }
  static __device__ __forceinline__ f32x4_t quad(const EMI_LDS uint8_t* lds, int q, int r) {
    return *reinterpret_cast<const EMI_LDS f32x4_t*>(lds + q * KP + slot(r) * 16);
  }
  static __device__ __forceinline__ bf16x8_t frag(const EMI_LDS uint8_t* lds, int plane, int piece, int r) {
    return *reinterpret_cast<const EMI_LDS bf16x8_t*>(lds + plane * PLANE + piece * KP + slot(r) * 16);
  }
};

// WM x WN wavefronts tile the block's BM x BN, or WM x WN x 2 where two share the k of a stage (WK == 2, added at the end).
// The LDS holds two stages: while t is multiplied, t + 1, loaded PF stages earlier, is split and laid out; one barrier a
// stage.  A wavefront alone issues an instruction of the split every 7.5 cycles, two on a SIMD every 3.7, and beside a
// matrix instruction every 9.5, so there are four on a SIMD, and the first half of them multiplies and then splits between two
// barriers, the other half splits and then multiplies: the arithmetic of the split runs beside the matrix cores.
// part != nullptr: split-K, split z owns the stages [z * steps_per_split, ...) of the contraction (of the whole sum, where
// products are summed) and leaves its tile in part[z][M][N] for the reduction over splits.
template <int BM, int BN, int WM, int WN, int WK, int PF, bool AKM, bool BKM, bool GROUPED>
__global__ __launch_bounds__(WM* WN* WK * 64, 4) void gemm_f32_split_kernel(const float* A, const float* B, const float* R, float* C, int M,
                                                                           int N, int K, int lda, int ldb, int64_t ldr, int64_t ldc,
                                                                           float* part, int steps_per_split,
                                                                           std::conditional_t<GROUPED, F32Group, F32Single> grp) {
  constexpr int BK = 32, NW = WM * WN * WK;
  constexpr int TM = BM / WM / 32, TN = BN / WN / 32;
  static_assert(WK == 1 || WK == 2, "a stage has two k-steps");
  using OA = SplitOperand<BM, NW * 64, PF, AKM>;
  using OB = SplitOperand<BN, NW * 64, PF, BKM>;
  constexpr int STAGE = OA::BYTES + OB::BYTES;
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem_raw[];
  EMI_LDS uint8_t* smem = (EMI_LDS uint8_t*)smem_raw;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 31, g = lane >> 5;
  const int wk = wave / (WM * WN), wm = wave % (WM * WN) / WN, wn = wave % WN;
  const bool late = wave >= NW / 2;                                // splits t + 1 before it multiplies t

  // workgroup ids go round the XCDs: give each XCD (own L2) a run of neighbouring tiles, eight tile rows deep, so that it
  // reads a few panels of both operands many times; splits and products outermost
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN, tiles = tiles_m * tiles_n;
  const int nb = gridDim.x, per = nb >> 3, rem = nb & 7, xcd = blockIdx.x & 7;
  const int pid = xcd * per + (xcd < rem ? xcd : rem) + (blockIdx.x >> 3);
  const int outer = pid / tiles, tile = pid - outer * tiles;
  const int first_m = tile / (8 * tiles_n) * 8, deep = tiles_m - first_m < 8 ? tiles_m - first_m : 8;
  const int in_group = tile - first_m * tiles_n;
  const int m0 = (first_m + in_group % deep) * BM, n0 = in_group / deep * BN;
  const int ksteps = (K + BK - 1) / BK;
  int step0 = 0, nsteps = ksteps;
  if constexpr (GROUPED) {
    if (grp.sum) {
      nsteps *= grp.count;
    } else {
      A = grp.A[outer];
      B = grp.B[outer];
      R = grp.R[outer];
      C = grp.C[outer];
    }
  }
  if (part != nullptr) {
    step0 = outer * steps_per_split;
    nsteps = nsteps - step0 < steps_per_split ? nsteps - step0 : steps_per_split;
    part += (int64_t)outer * M * N;
  }
  const int rows_a = M - m0 < BM ? M - m0 : BM, rows_b = N - n0 < BN ? N - n0 : BN;
  const int64_t a_row = AKM ? m0 : (int64_t)m0 * lda, b_row = BKM ? n0 : (int64_t)n0 * ldb;
  const int64_t a_k = AKM ? lda : 1, b_k = BKM ? ldb : 1;          // elements per k
  OA oa;
  OB ob;
  oa.init(rows_a, lda);
  ob.init(rows_b, ldb);

  int at_pair = 0, at_k = step0 * BK, to_load = nsteps;
  if constexpr (GROUPED) {
    if (grp.sum) {
      at_pair = step0 / ksteps;
      at_k = (step0 - at_pair * ksteps) * BK;
      A = grp.A[at_pair];
      B = grp.B[at_pair];
    }
  }
  auto load = [&](int f) __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);                             // in this order: the oldest stage is waited for, not all
    const int left = to_load-- > 0 ? K - at_k : 0;                 // past the last stage: zeros
    oa.load(f, A + a_row + at_k * a_k, rows_a, lda, left);
    ob.load(f, B + b_row + at_k * b_k, rows_b, ldb, left);
    at_k += BK;
    if constexpr (GROUPED) {
      if (at_k >= K && to_load > 0) {
        at_k = 0;
        at_pair++;
        A = grp.A[at_pair];
        B = grp.B[at_pair];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto sync = []() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

  constexpr f32x16_t zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  f32x16_t big[TM][TN], small[TM][TN], total[TM][TN];
#pragma unroll
  for (int a = 0; a < TM; a++)
#pragma unroll
    for (int b = 0; b < TN; b++) big[a][b] = small[a][b] = total[a][b] = zero;
  auto end_chain = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int a = 0; a < TM; a++)
#pragma unroll
      for (int b = 0; b < TN; b++) {
        total[a][b] += big[a][b] + small[a][b];
        big[a][b] = small[a][b] = zero;
      }
  };
  auto multiply = [&](const EMI_LDS uint8_t* s) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < 2 / WK; c++) {
      const int piece = 2 * (WK == 1 ? c : wk) + g;
      bf16x8_t fa[3][TM], fb[3][TN];
#pragma unroll
      for (int p = 0; p < 3; p++) {
#pragma unroll
        for (int a = 0; a < TM; a++) fa[p][a] = OA::frag(s, p, piece, wm * (BM / WM) + a * 32 + i);
#pragma unroll
        for (int b = 0; b < TN; b++) fb[p][b] = OB::frag(s + OA::BYTES, p, piece, wn * (BN / WN) + b * 32 + i);
      }
      auto add = [&](int p, int q, f32x16_t (&sum)[TM][TN]) __attribute__((always_inline)) {
#pragma unroll
        for (int a = 0; a < TM; a++)
#pragma unroll
          for (int b = 0; b < TN; b++) sum[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[p][a], fb[q][b], sum[a][b], 0, 0, 0);
      };
      add(0, 0, big);
      add(0, 1, small);
      add(1, 0, small);
      add(1, 1, small);
      add(0, 2, small);
      add(2, 0, small);
    }
  };
  auto store = [&](int f, int t) __attribute__((always_inline)) {    // (past the last stage: zeros, not multiplied)
    oa.store(f, smem + (t & 1) * STAGE);
    ob.store(f, smem + (t & 1) * STAGE + OA::BYTES);
  };

  load(PF);
  if (late) load(PF + 1);
#pragma unroll
  for (int f = 0; f < PF; f++) load(f);
  store(PF, 0);
  sync();
  if (late) store(PF + 1, 1);
  auto stage = [&](int t, int f) __attribute__((always_inline)) {
    __builtin_amdgcn_s_setprio(1);
    multiply(smem + (t & 1) * STAGE);
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
    if (late) sync();
    store(f, t + 1 + late);
    load(f);
    if (!late) sync();
  };
  // whole rounds of the PF stages in flight without a way out in between: where ways meet, the compiler waits for all loads
  int t = 0;
  for (; t + PF <= nsteps; t += PF) {
#pragma unroll
    for (int u = 0; u < PF; u++) stage(t + u, u);
    end_chain();
  }
#pragma unroll
  for (int u = 0; u < PF - 1; u++)
    if (t + u < nsteps) stage(t + u, u);
  end_chain();

  // Where the split does not hold, the tile is multiplied again in fp32 as it is, in stages through the LDS (us for the whole
  // product, ordinary numbers | all tiles again | the same on the fp32 kernels alone: 2000 x 768 x 768 26 | 56 | 33,
  // 777 x 4096 x 4096 162 | 428 | 232, 4096^3 730 | 1730 | 1008): a number that may not be the sum of its parts, and numbers that
  // are infinite, NaN or round to an infinite h (some sum is not finite then).
  bool odd = oa.inexact() || ob.inexact();
#pragma unroll
  for (int a = 0; a < TM; a++)
#pragma unroll
    for (int b = 0; b < TN; b++) {
      float z = 0.f;
#pragma unroll
      for (int r = 0; r < 16; r++) z = __builtin_fmaf(total[a][b][r], 0.f, z);
      odd = odd || z != 0.f;
    }
  EMI_LDS uint32_t* flags = (EMI_LDS uint32_t*)smem;
  const uint32_t seen = __any(odd);
  __syncthreads();
  if (lane == 0) flags[wave] = seen;
  __syncthreads();
  uint32_t again = 0;
#pragma unroll
  for (int w = 0; w < NW; w++) again |= flags[w];
  if (__builtin_amdgcn_readfirstlane(again) != 0) {
    __syncthreads();
    at_pair = 0, at_k = step0 * BK, to_load = nsteps;
    if constexpr (GROUPED) {
      if (grp.sum) {
        at_pair = step0 / ksteps;
        at_k = (step0 - at_pair * ksteps) * BK;
        A = grp.A[at_pair];
        B = grp.B[at_pair];
      }
    }
#pragma unroll
    for (int a = 0; a < TM; a++)
#pragma unroll
      for (int b = 0; b < TN; b++) total[a][b] = zero;
    load(0);
    for (int t = 0; t < nsteps; t++) {
      EMI_LDS uint8_t* s = smem + (t & 1) * STAGE;
      oa.store_f32(0, s);
      ob.store_f32(0, s + OA::BYTES);
      load(0);
      sync();                                                      // (the other stage is written once all are here again)
#pragma unroll
      for (int a = 0; a < TM; a++)
#pragma unroll
        for (int b = 0; b < TN; b++) big[a][b] = zero;
#pragma unroll
      for (int c = 0; c < 4 / WK; c++) {                           // eight k: the two halves of the wavefront have four each
        const int q = 2 * (wk * (4 / WK) + c) + g;
        f32x4_t fa[TM], fb[TN];
#pragma unroll
        for (int a = 0; a < TM; a++) fa[a] = OA::quad(s, q, wm * (BM / WM) + a * 32 + i);
#pragma unroll
        for (int b = 0; b < TN; b++) fb[b] = OB::quad(s + OA::BYTES, q, wn * (BN / WN) + b * 32 + i);
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
          for (int a = 0; a < TM; a++)
#pragma unroll
            for (int b = 0; b < TN; b++) big[a][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[a][e], fb[b][e], big[a][b], 0, 0, 0);
      }
#pragma unroll
      for (int a = 0; a < TM; a++)
#pragma unroll
        for (int b = 0; b < TN; b++) total[a][b] += big[a][b];
    }
    __syncthreads();
  }

  // register r of lane l: row 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32 of its 32 x 32 tile.  Of two wavefronts that
  // share k each finishes eight of the sixteen.
  if constexpr (WK == 2) {
    EMI_LDS float* mine = (EMI_LDS float*)(smem + 64) + (wave * TM * TN) * 8 * 64 + lane;
    const EMI_LDS float* theirs = (EMI_LDS float*)(smem + 64) + ((wave ^ (NW / 2)) * TM * TN) * 8 * 64 + lane;
    static_assert(64 + NW * TM * TN * 8 * 64 * 4 <= 2 * STAGE, "the exchange fits the stages");
#pragma unroll
    for (int a = 0; a < TM; a++)
#pragma unroll
      for (int b = 0; b < TN; b++)
#pragma unroll
        for (int r = 0; r < 8; r++) mine[((a * TN + b) * 8 + r) * 64] = wk == 0 ? total[a][b][8 + r] : total[a][b][r];
    __syncthreads();
#pragma unroll
    for (int a = 0; a < TM; a++)
#pragma unroll
      for (int b = 0; b < TN; b++)
#pragma unroll
        for (int r = 0; r < 8; r++) total[a][b][r] = (wk == 0 ? total[a][b][r] : total[a][b][8 + r]) + theirs[((a * TN + b) * 8 + r) * 64];
  }
  const int64_t ld = part != nullptr ? N : ldc;
  const bool add_r = part == nullptr && R != nullptr;
  auto window = [&](const float* base, int64_t row_length) __attribute__((always_inline)) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base) + m0 * row_length + n0, 0, (uint32_t)((rows_a - 1) * row_length + rows_b) * 4u,
                                             0x00020000);
  };
  const __amdgpu_buffer_rsrc_t to = window(part != nullptr ? part : C, ld), from = window(add_r ? R : C, add_r ? ldr : ld);
#pragma unroll
  for (int b = 0; b < TN; b++) {
    const int col = wn * (BN / WN) + b * 32 + i, row = wm * (BM / WM) + g * 4 + wk * 16;
    const bool in = col < rows_b;                                  // (rows past the last one lie past the window)
    uint32_t at_c = in ? (uint32_t)(row * (int)ld + col) * 4u : kOob, at_r = in ? (uint32_t)(row * (int)ldr + col) * 4u : kOob;
#pragma unroll
    for (int a = 0; a < TM; a++)
#pragma unroll
      for (int r = 0; r < 16 / WK; r++) {
        const int down = a * 32 + (r >> 2) * 8 + (r & 3);
        float v = total[a][b][r];
        if (add_r) v += __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(from, at_r + (uint32_t)(down * (int)ldr) * 4u, 0, 0));
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), to, at_c + (uint32_t)(down * (int)ld) * 4u, 0, 0);
      }
  }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

template <int BM, int BN, int WM, int WN, int WK, int PF, bool AKM, bool BKM, bool GROUPED>
static int launch_split_one(hipStream_t st, const F32Call& c) {
  auto kern = gemm_f32_split_kernel<BM, BN, WM, WN, WK, PF, AKM, BKM, GROUPED>;
  constexpr int smem = 2 * (SplitOperand<BM, WM * WN * WK * 64, PF, AKM>::BYTES + SplitOperand<BN, WM * WN * WK * 64, PF, BKM>::BYTES);
  static_assert(smem <= 160 * 1024, "LDS of a CU");
  static bool configured = false;   // idempotent; a race only repeats the call
  if (!configured) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    if (e != hipSuccess) return emi_fail(EMI_INTERNAL, "emi_gemm: cannot reserve %d bytes of LDS: %s", smem, hipGetErrorString(e));
    configured = true;
  }
  const int steps = ((c.K + 31) / 32) * (GROUPED && c.grp->sum ? c.grp->count : 1);
  const int sps = (steps + c.splits - 1) / c.splits, nz = (steps + sps - 1) / sps;
  const int outer = GROUPED && !c.grp->sum ? c.grp->count : nz;
  const int tiles = ((c.M + BM - 1) / BM) * ((c.N + BN - 1) / BN);
  float* part = outer == nz && nz > 1 ? c.part : nullptr;
  if constexpr (GROUPED)
    hipLaunchKernelGGL(kern, dim3(tiles * outer), dim3(WM * WN * WK * 64), smem, st, c.A, c.B, c.R, c.C, c.M, c.N, c.K, c.lda, c.ldb, c.ldr,
                       c.ldc, part, sps, *c.grp);
  else
    hipLaunchKernelGGL(kern, dim3(tiles * outer), dim3(WM * WN * WK * 64), smem, st, c.A, c.B, c.R, c.C, c.M, c.N, c.K, c.lda, c.ldb, c.ldr,
                       c.ldc, part, sps, F32Single{});
  EMI_CHECK_LAUNCH("emi_gemm(fp32)");
  if (part != nullptr && c.planes != nullptr) {
    *c.planes = nz;
    return EMI_OK;
  }
  if (part != nullptr) return launch_f32_splitk_reduce(st, part, c.R, c.C, c.M, c.N, nz, c.ldr, c.ldc);
  return EMI_OK;
}

template <int BM, int BN, int WM, int WN, int WK, int PF>
static int launch_split_shape(hipStream_t st, const F32Call& c, int trans_a, int trans_b) {
#define EMI_F32_SPLIT(AKM, BKM)                                                                             \
  return c.grp != nullptr ? launch_split_one<BM, BN, WM, WN, WK, PF, AKM, BKM, true>(st, c)                   \
                          : launch_split_one<BM, BN, WM, WN, WK, PF, AKM, BKM, false>(st, c)
  if (!trans_a && trans_b) EMI_F32_SPLIT(false, false);
  if (!trans_a && !trans_b) EMI_F32_SPLIT(false, true);
  if (trans_a && !trans_b) EMI_F32_SPLIT(true, true);
  EMI_F32_SPLIT(true, false);
#undef EMI_F32_SPLIT
}

int launch_f32_bf16x3(hipStream_t st, const F32Call& c, int shape, int trans_a, int trans_b) {
  switch (shape) {
    case 0: return launch_split_shape<128, 128, 4, 4, 1, 3>(st, c, trans_a, trans_b);
    case 1: return launch_split_shape<128, 64, 4, 2, 1, 2>(st, c, trans_a, trans_b);
    default: return launch_split_shape<64, 64, 2, 2, 2, 2>(st, c, trans_a, trans_b);
  }
}

}  // namespace emi
