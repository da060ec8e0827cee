// fp32 products on v_mfma_f32_32x32x2_f32, operands streamed global -> LDS: those of few stages or few tiles.  What has more
// of both runs on the bf16 instructions (gemm_f32_split.hip); f32_plan() draws the line.
//
//   C[M,N] = op(A) . op(B) [+ R]      fp32 throughout
//
// An fp32 matrix instruction keeps its SIMD's matrix core busy for 64 cycles and needs 512 bytes of operands, a quarter
// of what the LDS delivers in that time to four SIMDs.  On few tiles what counts is that loads are in flight all the time and
// that every CU has the same share of the work.  So: a ring of NST LDS stages of BK k each, filled by direct-to-LDS loads
// (16 bytes a lane, no staging registers) NST - 1 stages ahead, one barrier per stage, and blocks of 64 x 64, or of 32 x 32
// whose eight wavefronts share k (128 x 128 where a contraction is one stage).  Measured, us (NT / NN / TN form): 256 x 288 x 288 4.9 / 5.4 / 4.9; 256 x 288 x 768 7.3;
// 256 x 768 x 768 7.8.  What is left is the latency of the first loads and the launch.
#include <type_traits>

#include "emi_device.h"
#include "gemm_f32.h"
#include "gemm_plan.h"

namespace emi {

typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16_t;
#define EMI_LDS __attribute__((address_space(3)))
constexpr uint32_t kOob = 0x80000000u;   // beyond any buffer's num_records: loads return 0

template <int N> __device__ __forceinline__ void f32_wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0f70);
}

// One operand of a block: ROWS rows (of A: rows of C; of B: columns of C) by BK of the contraction per stage.
// k-contiguous (KM == false, stored [row][k]): LDS rows of BK floats, 16-byte piece c of row r at piece c ^ swz(r), which
// spreads the 16 rows that one pass of a ds_read_b128 serves over all banks.
// k-major (KM == true, stored [k][row]): LDS rows of ROWS floats.  A fragment read takes 32 consecutive columns of k-row
// 8j + t and of k-row 8j + 4 + t; pieces of a row with bit 2 of k set are stored 32 columns across (ROWS >= 64), or
// such a row takes its neighbour's place (ROWS == 32, two rows per bank line), so that the two do not share banks.
template <int ROWS, int BK, int NW, bool KM> struct F32Operand {
  static constexpr int BYTES = ROWS * BK * 4;
  static constexpr int LOADS = BYTES / 1024 / NW;                 // 1 KiB wave-loads per wavefront and stage
  static_assert(LOADS >= 1, "a stage is smaller than one pass of the block");
  static constexpr int CPR = (KM ? ROWS : BK) / 4;                // 16-byte pieces per LDS row
  static __device__ __forceinline__ int swz(int r) { return CPR == 8 ? ((r >> 1) & 7) : (r & 15); }

  // what this lane's it-th load of a stage fetches: byte offset from the stage's corner of the operand (kOob: outside)
  // and, k-contiguous, the k of its piece (k-major pieces past the contraction lie past num_records)
  uint32_t voff[LOADS];
  int lk[LOADS];
  __device__ __forceinline__ void init(int wave, int lane, int rows_left, int ld) {
#pragma unroll
    for (int it = 0; it < LOADS; it++) {
      const int slot = (it * NW + wave) * 64 + lane, r = slot / CPR, pc = slot % CPR;
      if constexpr (KM) {
        const int k = ROWS == 32 ? r ^ ((r >> 2) & 1) : r;
        const int col = (ROWS == 32 ? pc : pc ^ (8 * ((k >> 2) & 1))) * 4;
        lk[it] = 0;
        voff[it] = col < rows_left ? (uint32_t)(k * ld + col) * 4u : kOob;
      } else {
        lk[it] = (pc ^ swz(r)) * 4;
        voff[it] = r < rows_left ? (uint32_t)(r * ld + lk[it]) * 4u : kOob;
      }
    }
  }
  // corner: the operand at the block's first row and the stage's first k, of which `left` are left to contract
  __device__ __forceinline__ void issue(const float* corner, EMI_LDS uint8_t* lds, int wave, int rows, int ld, int left) const {
    const uint32_t bytes = left <= 0 ? 0u : (uint32_t)(KM ? ((left < BK ? left : BK) - 1) * ld + rows : (rows - 1) * ld + left) * 4u;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(corner), 0, bytes, 0x00020000);
#pragma unroll
    for (int it = 0; it < LOADS; it++) {
      const uint32_t v = KM || lk[it] < left ? voff[it] : kOob;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, lds + (it * NW + wave) * 1024, 16, v, 0, 0, 0);
    }
  }
  // the four k (8j + 4g .. + 3) of tile row `row` that this lane contracts
  static __device__ __forceinline__ void frag(const EMI_LDS uint8_t* lds, int row, int g, int j, float (&f)[4]) {
    if constexpr (KM) {
#pragma unroll
      for (int t = 0; t < 4; t++) {
        const int k = 8 * j + 4 * g + t;
        const int at = ROWS == 32 ? (k ^ g) * ROWS + row : k * ROWS + (row ^ (32 * g));
        f[t] = *reinterpret_cast<const EMI_LDS float*>(lds + at * 4);
      }
    } else {
      typedef __attribute__((__vector_size__(4 * sizeof(float)))) float v4;
      const v4 x = *reinterpret_cast<const EMI_LDS v4*>(lds + row * (BK * 4) + (((2 * j + g) ^ swz(row)) << 4));
      f[0] = x[0]; f[1] = x[1]; f[2] = x[2]; f[3] = x[3];
    }
  }
};

// WM x WN wavefronts tile the block's BM x BN; WK wavefronts share the k of every stage (chunk j of 8 to wavefront
// j % WK) and are added in wavefront order at the end.  The contraction index of an instruction is the lane half g:
// instruction t of chunk j contracts k = 8j + 4g + t, so that a k-contiguous operand is read in 16-byte pieces.
// part != nullptr: split-K, split z owns the stages [z * steps_per_split, ...) of the contraction (of the whole sum, where
// products are summed) and leaves its tile in part[z][M][N] for the reduction over splits.
// MODE (gemm_plan.h), beside a single product and a group: gated, the products with w1 and w3 one after the other in one block,
// whose tiles meet in the SwiGLU; rotated, up to three results, each lane exchanging its column with its neighbour's; adjoint,
// the SwiGLU's adjoint of the tile.  us,
// separate launches | this: gated 183 x 768 x 288 10.8 | 8.3, 308 x 1408 x 512 18.9 | 18.1; rotated, three results, 236 x 288 x 288 7.9 | 6.0,
// 62 x 768 x 768 11.1 | 8.7; adjoint 223 x 768 x 288 7.9 | 5.9, 198 x 1408 x 512 12.5 | 10.2.
template <int MODE> struct F32Arg { using type = F32Single; };
template <> struct F32Arg<kTailGroup> { using type = F32Group; };
template <> struct F32Arg<kTailGated> {
  struct type {
    const float* B1;
    float *C1, *G;
  };
};
template <> struct F32Arg<kTailRotated> {
  struct type {
    const float* B[3];
    float* C[3];
    const float2* table;
    int seq, head_dim, rotated, pairs;
    const float *A1, *B1[3];
  };
};
template <> struct F32Arg<kTailAdjoint> {
  struct type {
    const float *h1, *h3;
    float* d3;
  };
};
__device__ __forceinline__ float lane_xor1(float v) {
  return __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), 0xb1, 0xf, 0xf, true));
}

template <int BM, int BN, int WM, int WN, int WK, int BK, int NST, bool AKM, bool BKM, int MODE>
__global__ __launch_bounds__(WM* WN* WK * 64, 2) void gemm_f32_pipe_kernel(const float* A, const float* B, const float* R, float* C, int M,
                                                                        int N, int K, int lda, int ldb, int64_t ldr, int64_t ldc,
                                                                        float* part, int steps_per_split,
                                                                        typename F32Arg<MODE>::type grp) {
  constexpr bool GROUPED = MODE == kTailGroup;
  constexpr int NW = WM * WN * WK;
  constexpr int TM = BM / WM / 32, TN = BN / WN / 32;
  constexpr int CH = BK / 8 / WK;                                 // 8-wide chunks per wavefront and stage
  static_assert(WK == 1 || (TM == 1 && TN == 1 && WM == 1 && WN == 1), "wavefronts share k on a single 32 x 32 tile");
  static_assert(NST >= 2 && CH >= 1, "stages");
  using OA = F32Operand<BM, BK, NW, AKM>;
  using OB = F32Operand<BN, BK, NW, BKM>;
  constexpr int STAGE = OA::BYTES + OB::BYTES;
  constexpr int LPT = OA::LOADS + OB::LOADS;
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem_raw[];
  EMI_LDS uint8_t* smem = (EMI_LDS uint8_t*)smem_raw;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 31, g = lane >> 5;
  const int wk = WK == 1 ? 0 : wave, wm = WK == 1 ? wave / WN : 0, wn = WK == 1 ? wave % WN : 0;

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
  if constexpr (MODE == kTailGated) nsteps *= 2;
  if constexpr (MODE == kTailRotated) {
    B = grp.B[outer];
    C = grp.C[outer];
    nsteps *= grp.pairs;
  }
  if (part != nullptr) {
    step0 = outer * steps_per_split;
    nsteps = nsteps - step0 < steps_per_split ? nsteps - step0 : steps_per_split;
    part += (int64_t)outer * M * N;
  }
  const int rows_a = M - m0 < BM ? M - m0 : BM, rows_b = N - n0 < BN ? N - n0 : BN;
  OA oa;
  OB ob;
  oa.init(wave, lane, rows_a, lda);
  ob.init(wave, lane, rows_b, ldb);
  const int64_t a_row = AKM ? m0 : (int64_t)m0 * lda, b_row = BKM ? n0 : (int64_t)n0 * ldb;
  const int64_t a_k = AKM ? lda : 1, b_k = BKM ? ldb : 1;          // elements per k

  // stages in issue order; past the last one the loads still go out (as zeros) so that the number in flight is constant
  int at_pair = 0, at_k = step0 * BK, at_slot = 0, to_issue = nsteps;
  if constexpr (GROUPED) {
    if (grp.sum) {
      at_pair = step0 / ksteps;
      at_k = (step0 - at_pair * ksteps) * BK;
      A = grp.A[at_pair];
      B = grp.B[at_pair];
    }
  }
  auto issue = [&]() __attribute__((always_inline)) {
    const int left = to_issue-- > 0 ? K - at_k : 0;
    EMI_LDS uint8_t* s = smem + at_slot * STAGE;
    oa.issue(A + a_row + at_k * a_k, s, wave, rows_a, lda, left);
    ob.issue(B + b_row + at_k * b_k, s + OA::BYTES, wave, rows_b, ldb, left);
    at_slot = at_slot + 1 < NST ? at_slot + 1 : 0;
    at_k += BK;
    if constexpr (GROUPED) {
      if (at_k >= K && to_issue > 0) {
        at_k = 0;
        at_pair++;
        A = grp.A[at_pair];
        B = grp.B[at_pair];
      }
    }
    if constexpr (MODE == kTailGated) {
      if (at_k >= K) {
        at_k = 0;
        B = grp.B1;
      }
    }
    if constexpr (MODE == kTailRotated) {
      if (at_k >= K && to_issue > 0) {
        at_k = 0;
        A = grp.A1;
        B = grp.B1[outer];
      }
    }
  };

  // A sum over K in one chain is off by the square root of its length, so a chain ends after FLUSH stages (32 k of a
  // wavefront, 64 where wavefronts share k) and goes into `total`; after every stage that happens while the next one's
  // fragments are on their way.  2 % of the time; relative error of 2048 x 768 x 2000 5.7e-7 -> 1.5e-7.
  constexpr int FLUSH = WK > 1 ? 8 : 1;
  constexpr f32x16_t zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  f32x16_t acc[TM][TN], total[TM][TN];
#pragma unroll
  for (int a = 0; a < TM; a++)
#pragma unroll
    for (int b = 0; b < TN; b++) acc[a][b] = total[a][b] = zero;
  auto end_chain = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int a = 0; a < TM; a++)
#pragma unroll
      for (int b = 0; b < TN; b++) {
        total[a][b] += acc[a][b];
        acc[a][b] = zero;
      }
  };

  // Which element of the result this lane's e-th is.  Wavefronts that share k meet in the LDS; otherwise register r of lane l
  // holds row 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32 of its 32 x 32 tile.
  constexpr int EACH = WK > 1 ? 1024 / (NW * 64) : 16 * TM * TN;
  auto row_of = [&](int e) __attribute__((always_inline)) {
    if constexpr (WK > 1) return m0 + ((e * NW * 64 + (int)threadIdx.x) >> 5);
    else return m0 + wm * (BM / WM) + e / (16 * TN) * 32 + (e % 16 >> 2) * 8 + g * 4 + (e & 3);
  };
  auto col_of = [&](int e) __attribute__((always_inline)) {
    if constexpr (WK > 1) return n0 + ((e * NW * 64 + (int)threadIdx.x) & 31);
    else return n0 + wn * (BN / WN) + e / 16 % TN * 32 + i;
  };
  // What an elementwise operator needs beside the product is requested ahead of the ring's loads: after the contraction, each
  // load behind the stores before it, it cost 4 to 8 us (64 x 64 blocks).
  [[maybe_unused]] float beside[2][EACH];
  if constexpr (MODE == kTailRotated || MODE == kTailAdjoint) {
#pragma unroll
    for (int e = 0; e < EACH; e++) {
      const int row = row_of(e) < M ? row_of(e) : M - 1, col = col_of(e) < N ? col_of(e) : N - 1;
      if constexpr (MODE == kTailAdjoint) {
        const int64_t at = (int64_t)row * ldc + col;
        beside[0][e] = grp.h1[at];
        beside[1][e] = grp.h3[at];
      } else {
        const float2 t = outer < grp.rotated ? grp.table[(int64_t)(row % grp.seq) * (grp.head_dim >> 1) + ((col % grp.head_dim) >> 1)] : make_float2(1.f, 0.f);
        beside[0][e] = t.x;
        beside[1][e] = t.y;
      }
    }
  }

#pragma unroll
  for (int s = 0; s < NST - 1; s++) issue();
  int slot = 0;
  auto stage = [&]() __attribute__((always_inline)) {
    f32_wait_vmcnt<(NST - 2) * LPT>();                     // this stage has landed
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();                          // everyone's part of it, and the stage before is free again
    __builtin_amdgcn_sched_barrier(0);
    issue();
    const EMI_LDS uint8_t* sa = smem + slot * STAGE;
    const EMI_LDS uint8_t* sb = sa + OA::BYTES;
    slot = slot + 1 < NST ? slot + 1 : 0;
    float fa[2][TM][4], fb[2][TN][4];
    auto read = [&](int c, float (&pa)[TM][4], float (&pb)[TN][4]) __attribute__((always_inline)) {
      const int j = c * WK + wk;
#pragma unroll
      for (int a = 0; a < TM; a++) OA::frag(sa, wm * (BM / WM) + a * 32 + i, g, j, pa[a]);
#pragma unroll
      for (int b = 0; b < TN; b++) OB::frag(sb, wn * (BN / WN) + b * 32 + i, g, j, pb[b]);
    };
    read(0, fa[0], fb[0]);
    if constexpr (FLUSH == 1) end_chain();                // of the stage before
#pragma unroll
    for (int c = 0; c < CH; c++) {
      if (c + 1 < CH) read(c + 1, fa[(c + 1) & 1], fb[(c + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);                   // the next chunk's reads stay ahead of this one's products
#pragma unroll
      for (int q = 0; q < 4; q++)
#pragma unroll
        for (int a = 0; a < TM; a++)
#pragma unroll
          for (int b = 0; b < TN; b++)
            acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[c & 1][a][q], fb[c & 1][b][q], acc[a][b], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto contract = [&](int steps) __attribute__((always_inline)) {
    for (int t = 0; t < steps;) {
      if constexpr (FLUSH > 1) {
#pragma unroll 1
        for (const int end = t + FLUSH < steps ? t + FLUSH : steps; t < end; t++) stage();
        end_chain();
      } else {
        stage();
        t++;
      }
    }
    if constexpr (FLUSH == 1) end_chain();
  };
  f32x16_t gate[TM][TN];                                   // gated: the tile of h1
  if constexpr (MODE == kTailGated) {
    contract(ksteps);
#pragma unroll
    for (int a = 0; a < TM; a++)
#pragma unroll
      for (int b = 0; b < TN; b++) {
        gate[a][b] = total[a][b];
        total[a][b] = zero;
      }
    contract(ksteps);
  } else {
    contract(nsteps);
  }

  // element e of this lane's: what the elementwise operator reads beside it has been there since before the contraction
  auto put = [&](int row, int col, float v, float h1, float p, float q) __attribute__((always_inline)) {
    if constexpr (MODE == kTailRotated) {                  // the pair's other column is the neighbouring lane's, of the same row
      if (outer < grp.rotated) {                           // (turned by no angle, an infinity would make its neighbour a NaN)
        const float other = lane_xor1(v);
        v = (col & 1) == 0 ? rotated_even(p, q, v, other) : rotated_odd<float>(p, q, other, v);
      }
    }
    if (row < M && col < N) {
      if (part != nullptr) {
        part[(int64_t)row * N + col] = v;
      } else if constexpr (MODE == kTailGated) {
        const int64_t at = (int64_t)row * ldc + col;
        C[at] = h1;
        grp.C1[at] = v;
        grp.G[at] = emi_swiglu(h1, v);
      } else if constexpr (MODE == kTailAdjoint) {
        const int64_t at = (int64_t)row * ldc + col;
        float d1, d3;
        emi_swiglu_adjoint(p, q, v, &d1, &d3);
        C[at] = d1;
        grp.d3[at] = d3;
      } else {
        if (R != nullptr) v += R[(int64_t)row * ldr + col];
        C[(int64_t)row * ldc + col] = v;
      }
    }
  };
  f32_wait_vmcnt<0>();                                     // the zero-filled loads past the end
  if constexpr (WK > 1) {
    EMI_LDS float* red = (EMI_LDS float*)smem;             // [WK][32][32 + 1]
    float sum[EACH], h1[EACH];
    auto meet = [&](const f32x16_t& t) __attribute__((always_inline)) {
      __syncthreads();
#pragma unroll
      for (int r = 0; r < 16; r++) red[(wk * 32 + (r >> 2) * 8 + g * 4 + (r & 3)) * 33 + i] = t[r];
      __syncthreads();
#pragma unroll
      for (int e = 0; e < EACH; e++) {
        const int at = e * NW * 64 + threadIdx.x, row = at >> 5, col = at & 31;
        sum[e] = 0.f;
#pragma unroll
        for (int w = 0; w < WK; w++) sum[e] += red[(w * 32 + row) * 33 + col];
      }
    };
    if constexpr (MODE == kTailGated) {
      meet(gate[0][0]);
#pragma unroll
      for (int e = 0; e < EACH; e++) h1[e] = sum[e];
    }
    meet(total[0][0]);
#pragma unroll
    for (int e = 0; e < EACH; e++) put(row_of(e), col_of(e), sum[e], h1[e], beside[0][e], beside[1][e]);
  } else {
#pragma unroll
    for (int e = 0; e < EACH; e++) {
      const int a = e / (16 * TN), b = e / 16 % TN, r = e % 16;
      put(row_of(e), col_of(e), total[a][b][r], gate[a][b][r], beside[0][e], beside[1][e]);
    }
  }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

template <int BM, int BN, int WM, int WN, int WK, int BK, int NST, bool AKM, bool BKM, bool GROUPED>
static int launch_f32_one(hipStream_t st, const F32Call& c) {
  auto kern = gemm_f32_pipe_kernel<BM, BN, WM, WN, WK, BK, NST, AKM, BKM, GROUPED ? kTailGroup : kTailNone>;
  constexpr int smem = NST * (BM + BN) * BK * 4;
  static_assert(WK == 1 || smem >= WK * 32 * 33 * 4, "the wavefronts' tiles meet in the ring");
  static bool configured = false;
  if (const int rc = reserve_lds(reinterpret_cast<const void*>(kern), smem, configured)) return rc;
  const int steps = ((c.K + BK - 1) / BK) * (GROUPED && c.grp->sum ? c.grp->count : 1);
  const int sps = (steps + c.splits - 1) / c.splits, nz = (steps + sps - 1) / sps;
  const int outer = GROUPED && !c.grp->sum ? c.grp->count : nz;
  const int tiles = ((c.M + BM - 1) / BM) * ((c.N + BN - 1) / BN);
  float* part = outer == nz && nz > 1 ? c.part : nullptr;
  if constexpr (GROUPED)
    hipLaunchKernelGGL(kern, dim3(tiles * outer), dim3(WM * WN * WK * 64), smem, st, c.A, c.B, c.R, c.C, c.M, c.N, c.K, c.lda, c.ldb,
                       c.ldr, c.ldc, part, sps, *c.grp);
  else
    hipLaunchKernelGGL(kern, dim3(tiles * outer), dim3(WM * WN * WK * 64), smem, st, c.A, c.B, c.R, c.C, c.M, c.N, c.K, c.lda, c.ldb,
                       c.ldr, c.ldc, part, sps, F32Single{});
  EMI_CHECK_LAUNCH("emi_gemm(fp32)");
  if (part != nullptr && c.planes != nullptr) {
    *c.planes = nz;
    return EMI_OK;
  }
  if (part != nullptr) return launch_f32_splitk_reduce(st, part, c.R, c.C, c.M, c.N, nz, c.ldr, c.ldc);
  return EMI_OK;
}

template <int BM, int BN, int WM, int WN, int WK, int BK, int NST>
static int launch_f32_shape(hipStream_t st, const F32Call& c, int trans_a, int trans_b) {
#define EMI_F32_PIPE(AKM, BKM)                                                                          \
  return c.grp != nullptr ? launch_f32_one<BM, BN, WM, WN, WK, BK, NST, AKM, BKM, true>(st, c)          \
                          : launch_f32_one<BM, BN, WM, WN, WK, BK, NST, AKM, BKM, false>(st, c)
  if (!trans_a && trans_b) EMI_F32_PIPE(false, false);
  if (!trans_a && !trans_b) EMI_F32_PIPE(false, true);
  if (trans_a && !trans_b) EMI_F32_PIPE(true, true);
  EMI_F32_PIPE(true, false);
#undef EMI_F32_PIPE
}

// Which block and how many splits.  The estimate is of the CU with the most blocks, in microseconds: a start, which grows
// with the blocks that come after one another, and the stages at the rate of each block shape; a stage on the bf16 instructions
// takes longer the more blocks the chip has per CU, as its clock falls while it fills, and of a k-major A.  Fitted to 4000
// products of 16 to 4096 tokens by weights of 288 x 288 to 4096 x 11008, 64 MB of them in turn from beyond the L2s, each with the
// blocks and splits that could be the fastest: 0.2 % behind the fastest of them in the geometric mean and 14 % at the worst
// (0.9 and 26 % with rates taken at a few sizes with operands in the caches).  The fp32 blocks of 128 x 128 are for weight
// gradients of one stage: 12 of 1024 x 1024 x 19 17.8 us, 18.9 in blocks of 64 x 64, four of 2048 x 2048 x 24 21.6 | 23.4.
// The fp32 instructions keep what has few stages or few rows, us, the better of their blocks | of the others: 256 x 768 x 768
// 7.8 | 16, 840 x 768 x 768 17.2 | 18.4, 362 x 2048 x 768 17.5 | 19.5, 768 x 2048 x 36 (TN) 6.7 | 7.3; and beyond: 693 x 768 x 768 17.1 | 17.1,
// 1136 x 768 x 768 19.9 | 19.6, 2056 x 768 x 768 30.9 | 26.1, 180 x 11008 x 4096 167 | 137, 3122 x 768 x 288 (two) 33.8 | 29.
// The reduction over splits is a launch of its own; results over 4 M elements, whose planes leave the caches, and the products of
// a few tokens, which have kernels of their own (gemm_skinny.hip), are not split; a few rows of a k-major A are no such product
// (4 x 64 x 20000, us: 126 in one pass, 12 split).
struct F32Shape { int bm, bn, bk; };
constexpr int kF32Shapes = 6;                             // three of the fp32 instructions, three of the bf16
static const F32Shape kF32Shape[kF32Shapes] = {{64, 64, 32}, {32, 32, 64}, {128, 128, 32}, {128, 128, 32}, {128, 64, 32}, {64, 64, 32}};

// Microseconds of the products in blocks of shape c over z splits; not finite where it cannot be.
static double f32_estimate(int c, int64_t M, int64_t N, int64_t K, int count, int sum, int trans_a, int64_t z) {
  struct Fp32 { double one, base, block, rate[4]; };      // start of one block, of b: base + b block; rate[b - 1]: per stage, b blocks on
                                                          // the CU; the last one per block
  static const Fp32 fp32[3] = {{3.4, 3.25, 0.75, {0.68, 1.10, 1.615, 0.496}}, {3.2, 2.1, 1.16, {0.405, 0.69, 0.995, 0.35}},
                               {6.3, 4.0, 2.3, {2.01, 3.76, 5.94, 1.95}}};
  struct Bf16 { double base, block, one, one_fill, rate, fill; };        // per stage, one block on the CU | each of several; _fill: times blocks per CU of the chip
  static const Bf16 bf16[3] = {{3.2, 4.35, 0.76, 0.59, 0.975, 0.377}, {3.6, 1.6, 0.687, 0.228, 0.532, 0.25}, {2.3, 2.15, 0.511, 0.159, 0.359, 0.128}};
  const F32Shape& s = kF32Shape[c];
  const int64_t steps = (K + s.bk - 1) / s.bk * (sum ? count : 1);
  const int64_t blocks = (M + s.bm - 1) / s.bm * ((N + s.bn - 1) / s.bn) * (sum ? 1 : count);
  if (blocks > 0x3fffffff || (z > 1 && steps < 4 * z)) return 1e30;
  const int64_t b = (blocks * z + 255) / 256, per = (steps + z - 1) / z;
  const double several = count > 1 && !sum ? 0.6 : 0.0;   // results in one launch
  if (c < 3) {
    const Fp32& r = fp32[c];
    return (b == 1 ? r.one : r.base + r.block * b) + several + per * (b < 4 ? r.rate[b - 1] : r.rate[3] * b) +
           (z > 1 ? 2.8 + 1e-6 * M * N * (z + 1) : 0.0);
  }
  const Bf16& r = bf16[c - 3];
  const double stage = (b == 1 ? r.one : r.rate * b) + (b == 1 ? r.one_fill : r.fill) * (blocks * z / 256.0);
  return r.base + r.block * b + several + (trans_a ? 1.06 : 1.0) * per * stage + (z > 1 ? 3.7 + 0.5e-6 * M * N * (z + 1) : 0.0);
}

F32Plan f32_plan(int64_t M, int64_t N, int64_t K, int count, int sum, int trans_a, int64_t most) {
  F32Plan best{1, 1, 0.0};
  const bool may_split = (sum || count == 1) && M * N <= (4 << 20) && (M > 8 || trans_a) && K > 8;
  double least = 1e30;
  for (int c = 0; c < kF32Shapes; c++)
    for (int64_t z = 1; z <= (may_split ? 64 : 1) && z <= most; z++) {
      const double t = f32_estimate(c, M, N, K, count, sum, trans_a, z);
      if (t < least) {
        least = t;
        best = F32Plan{c, (int)z, t};
      }
    }
  return best;
}

size_t gemm_f32_workspace_bytes(int64_t M, int64_t N, int64_t K, int count, int sum, int trans_a) {
  const int z = f32_plan(M, N, K, count, sum, trans_a, kAnySplits).splits;
  return z > 1 ? (size_t)z * M * N * sizeof(float) : 0;
}

// C[i] = op(A[i]) . op(B[i]) [+ R[i]] for i < count, or with `sum` the one sum of the products (+ R[0]).  Returns -1 for
// operands that the kernels' 16-byte pieces do not fit (the caller has other kernels for those).
int launch_f32_gemm(hipStream_t st, int count, const void* const* A, const void* const* B, const void* const* R, void* const* C,
                    void* workspace, size_t workspace_bytes, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldr,
                    int64_t ldc, int trans_a, int trans_b, int sum, int* planes) {
  // pieces are four elements along the stored rows; a stage's panel of an operand is addressed with 31 bits
  if (K <= 0 || count > kMaxF32Group || lda % 4 || ldb % 4 || (trans_a ? M : K) % 4 || (trans_b ? K : N) % 4 ||
      128 * lda + K >= 0x1fffffff || 128 * ldb + K >= 0x1fffffff)
    return -1;
  F32Group g{};
  for (int i = 0; i < count; i++) {
    if ((reinterpret_cast<uintptr_t>(A[i]) | reinterpret_cast<uintptr_t>(B[i])) & 15) return -1;
    g.A[i] = static_cast<const float*>(A[i]);
    g.B[i] = static_cast<const float*>(B[i]);
  }
  for (int i = 0; i < (sum ? 1 : count); i++) {
    g.R[i] = R != nullptr ? static_cast<const float*>(R[i]) : nullptr;
    g.C[i] = static_cast<float*>(C[i]);
  }
  g.count = count;
  g.sum = sum;
  const int64_t held = splits_held(workspace, workspace_bytes, M, N);
  const F32Plan p = f32_plan(M, N, K, count, sum, trans_a, held);
  if (count > 1 && !sum && faster_one_by_one(p, f32_plan(M, N, K, 1, 0, trans_a, held), count, 1.0)) {
    for (int i = 0; i < count; i++) {
      const void* r = R != nullptr ? R[i] : nullptr;
      if (const int rc = launch_f32_gemm(st, 1, A + i, B + i, &r, C + i, workspace, workspace_bytes, M, N, K, lda, ldb, ldr, ldc, trans_a, trans_b, 0, nullptr))
        return rc;
    }
    return EMI_OK;
  }
  const F32Call c{g.A[0], g.B[0], g.R[0], g.C[0], (int)M, (int)N, (int)K, (int)lda, (int)ldb, ldr, ldc, static_cast<float*>(workspace),
                  p.splits, count > 1 ? &g : nullptr, planes};
  // (the split kernels address a tile of the result with 31 bits too)
  const bool wide = 128 * ldc >= 0x1fffffff || 128 * N >= 0x1fffffff || (R != nullptr && 128 * ldr >= 0x1fffffff);
  switch (wide && p.shape > 2 ? 0 : p.shape) {
    case 0: return launch_f32_shape<64, 64, 2, 2, 1, 32, 2>(st, c, trans_a, trans_b);
    case 1: return launch_f32_shape<32, 32, 1, 1, 8, 64, 5>(st, c, trans_a, trans_b);
    case 2: return launch_f32_shape<128, 128, 4, 2, 1, 32, 2>(st, c, trans_a, trans_b);
    default: return launch_f32_bf16x3(st, c, p.shape - 3, trans_a, trans_b);
  }
}

// The products of gemm_plan.h whose result goes through an elementwise operator, on the fp32 instructions.
template <int BM, int BN, int WM, int WN, int WK, int BK, int NST, bool BKM, int MODE>
static int launch_f32_tail_one(hipStream_t st, const float* A, const float* B, const ProductTail& t, int M, int N, int K, int ldb) {
  auto kern = gemm_f32_pipe_kernel<BM, BN, WM, WN, WK, BK, NST, false, BKM, MODE>;
  constexpr int smem = NST * (BM + BN) * BK * 4;
  static bool configured = false;
  if (const int rc = reserve_lds(reinterpret_cast<const void*>(kern), smem, configured)) return rc;
  typename F32Arg<MODE>::type arg{};
  if constexpr (MODE == kTailGated) {
    arg = {static_cast<const float*>(t.B[1]), static_cast<float*>(t.C[1]), static_cast<float*>(t.C[2])};
  } else if constexpr (MODE == kTailRotated) {
    for (int i = 0; i < t.count; i++) {
      arg.B[i] = static_cast<const float*>(t.B[i]);
      arg.C[i] = static_cast<float*>(t.C[i]);
      arg.B1[i] = static_cast<const float*>(t.B1[i]);
    }
    arg.A1 = static_cast<const float*>(t.A1);
    arg.pairs = t.A1 != nullptr ? 2 : 1;
    arg.table = reinterpret_cast<const float2*>(t.table);
    arg.seq = t.seq, arg.head_dim = t.head_dim, arg.rotated = t.rotated;
  } else {
    arg = {static_cast<const float*>(t.h1), static_cast<const float*>(t.h3), static_cast<float*>(t.C[1])};
  }
  const int tiles = ((M + BM - 1) / BM) * ((N + BN - 1) / BN) * (MODE == kTailRotated ? t.count : 1);
  hipLaunchKernelGGL(kern, dim3(tiles), dim3(WM * WN * WK * 64), smem, st, A, B, (const float*)nullptr, static_cast<float*>(t.C[0]), M, N, K, K,
                     ldb, (int64_t)0, (int64_t)N, (float*)nullptr, 0, arg);
  EMI_CHECK_LAUNCH("emi_gemm(fp32, elementwise tail)");
  return EMI_OK;
}
template <int BM, int BN, int WM, int WN, int WK, int BK, int NST>
static int launch_f32_tail_shape(hipStream_t st, const float* A, const float* B, const ProductTail& t, int M, int N, int K, int ldb, int trans_b) {
  if (t.mode == kTailGated) return launch_f32_tail_one<BM, BN, WM, WN, WK, BK, NST, false, kTailGated>(st, A, B, t, M, N, K, ldb);
  if (t.mode == kTailRotated) return launch_f32_tail_one<BM, BN, WM, WN, WK, BK, NST, false, kTailRotated>(st, A, B, t, M, N, K, ldb);
  return trans_b ? launch_f32_tail_one<BM, BN, WM, WN, WK, BK, NST, false, kTailAdjoint>(st, A, B, t, M, N, K, ldb)
                 : launch_f32_tail_one<BM, BN, WM, WN, WK, BK, NST, true, kTailAdjoint>(st, A, B, t, M, N, K, ldb);
}

// Against the separate launches by the plan's own estimates, and a pass of 2.4 us and the bytes it moves.  Gated, a block's two
// products cost what a sum of two does; a block's elementwise part, 0.8 us of a 32 x 32 tile and 3 of 64 x 64.  What has tiles and
// stages enough stays with the bf16 instructions and a pass (1970 x 2048 x 768 adjoint 56 | 63 here).
int launch_f32_tail(hipStream_t st, const void* A, const void* B, const ProductTail& t, int64_t M, int64_t N, int64_t K, int64_t ldb, int trans_b) {
  if (128 * K + K >= 0x1fffffff || 128 * ldb + K >= 0x1fffffff || (t.mode != kTailAdjoint && !trans_b)) return -1;
  const int count = t.mode == kTailGated ? 2 : t.mode == kTailRotated ? t.count : 1;
  const int pairs = t.A1 != nullptr ? 2 : 1;
  double together[2];
  for (int c = 0; c < 2; c++) {
    const int64_t blocks = (M + kF32Shape[c].bm - 1) / kF32Shape[c].bm * ((N + kF32Shape[c].bn - 1) / kF32Shape[c].bn) * (t.mode == kTailRotated ? count : 1);
    together[c] = f32_estimate(c, M, N, K * pairs, count, t.mode == kTailGated, 0, 1) + (c == 0 ? 3.0 : 0.8) * ((blocks + 255) / 256);
  }
  const int shape = together[1] < together[0];
  const double moved = 4e-6 / 5.0 * M * N * (t.mode == kTailRotated ? 2 * t.rotated : t.mode == kTailGated ? 3 : 5);
  // (two products to a result: each result would be a launch that sums them)
  const double apart = pairs == 2 ? count * (f32_plan(M, N, K, 2, 1, 0, kAnySplits).us + 1.0) : f32_plan(M, N, K, count, 0, 0, count > 1 ? 1 : kAnySplits).us;
  if (together[shape] >= apart + (t.mode == kTailRotated && t.rotated == 0 ? 0.0 : 2.4 + moved)) return -1;
  const float *a = static_cast<const float*>(A), *b = static_cast<const float*>(B);
  return shape == 0 ? launch_f32_tail_shape<64, 64, 2, 2, 1, 32, 2>(st, a, b, t, (int)M, (int)N, (int)K, (int)ldb, trans_b)
                    : launch_f32_tail_shape<32, 32, 1, 1, 8, 64, 5>(st, a, b, t, (int)M, (int)N, (int)K, (int)ldb, trans_b);
}

}  // namespace emi
