// bf16 products that do not fill the chip with the large tiles of gemm.hip: few tokens, or narrow results.
//
//   C[M,N] = A . op(B) [+ R]      A k-contiguous, fp32 accumulate, one rounding at the end
//
// What bounds these is not the matrix cores but the latency of a stage: the loads of a 128 x 128 tile that are in flight
// while one stage is multiplied cover 8 TB/s over the chip, and with few tiles most CUs have nothing else to do.  So, as in
// gemm_f32.hip: a ring of NST LDS stages filled by direct-to-LDS loads NST - 1 stages ahead, one barrier per stage, blocks
// from 128 x 128 down to 32 x 32 (whose eight wavefronts share k), and a launcher that chooses by how the tiles divide over
// the CUs (bf16_plan).  Eight wavefronts of 32 x 64 on a 128 x 128 tile read 1.5 times the LDS bytes of four of 64 x 64 and
// are still faster: two of them on a SIMD hide each other's LDS and barrier latency.
// Measured with all operands in the caches, us, against the two-stage 128 x 128 kernel of gemm.hip (k-contiguous B): 777 x 768 x 768 12.2 -> 5.5;
// 777 x 768 x 2048 18.7 -> 9.0; 64 x 768 x 768 9.9 -> 4.2; 300 x 5632 x 2048 23.2 -> 13.2; 1000 x 4096 x 4096 47.5 -> 37.0;
// 8192 x 768 x 768 15.4 -> 15.2, x 2048 30.5 -> 29.1; 8192 x 2304 x 768 42.4 -> 37.1 (782 TFLOP/s); k-major B:
// 777 x 768 x 768 15.5 -> 5.8; 1000 x 4096 x 4096 64.4 -> 36.6; 8192 x 768 x 2048 36.6 -> 30.4.  With weights from beyond the
// L2s, as a model has them: 777 x 768 x 768 5.9, x 2048 9.5, 512 x 1024 x 1024 6.5, 300 x 5632 x 2048 14.6, 1000 x 2048 x 2048 13.7,
// 1000 x 4096 x 4096 36.6, 8192 x 768 x 768 15.4, x 2048 29.6.
#include <type_traits>
#include <utility>

#include "emi_device.h"
#include "gemm_plan.h"

namespace emi {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
#define EMI_LDS __attribute__((address_space(3)))
constexpr uint32_t kOob = 0x80000000u;   // beyond any buffer's num_records: loads return 0

constexpr int kMaxPipeGroup = 48;
struct PipeGroup {
  const uint16_t* A[kMaxPipeGroup];
  const uint16_t* B[kMaxPipeGroup];
  const uint16_t* R[kMaxPipeGroup];
  uint16_t* C[kMaxPipeGroup];
  int count, sum;
};
struct PipeSingle {};

template <int N> __device__ __forceinline__ void pipe_wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0f70);
}
template <int OFF> __device__ __forceinline__ u32x2_t pipe_tr_read(uint32_t addr) {
  static_assert(OFF >= 0 && OFF < 65536, "ds offset field");
  u32x2_t r;
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(OFF));
  return r;
}

// One operand of a block: ROWS rows (of A: rows of C; of B: columns of C) by BK of the contraction per stage.
// k-contiguous (KM == false, stored [row][k]): LDS rows of BK elements, 16-byte piece c of row r at piece c ^ swz(r): the
// 16 rows that one pass of a ds_read_b128 serves lie on different banks.
// k-major (KM == true, stored [k][row]): LDS rows of ROWS elements read with the transposing LDS load; piece c of k-row k
// at c ^ kswz(k): the eight k-rows x 32 bytes that one pass of it serves (k = 0..3 and 8..11) lie on different banks.
template <int ROWS, int BK, int NW, bool KM> struct PipeOperand {
  static constexpr int BYTES = ROWS * BK * 2;
  static constexpr int LOADS = BYTES / 1024 / NW;                 // 1 KiB wave-loads per wavefront and stage
  static_assert(LOADS >= 1 && BYTES % (1024 * NW) == 0, "a stage is not a whole number of passes of the block");
  static constexpr int CPR = (KM ? ROWS : BK) / 8;                // 16-byte pieces per LDS row
  static_assert(!KM || ROWS == 64 || ROWS == 128, "k-major tiles are 64 or 128 wide");
  static __device__ __forceinline__ int swz(int r) { return CPR == 8 ? ((r >> 1) & 7) : (r & 15); }
  static __device__ __forceinline__ int kswz(int k) {
    return ROWS == 64 ? 2 * (((k >> 1) & 1) | (((k >> 3) & 1) << 1)) : (4 * (k & 3)) ^ (2 * ((k >> 3) & 1));
  }
  uint32_t voff[LOADS];
  int lk[LOADS];
  __device__ __forceinline__ void init(int wave, int lane, int rows_left, int ld) {
#pragma unroll
    for (int it = 0; it < LOADS; it++) {
      const int slot = (it * NW + wave) * 64 + lane, r = slot / CPR, pc = slot % CPR;
      if constexpr (KM) {
        const int col = (pc ^ kswz(r)) * 8;
        lk[it] = 0;
        voff[it] = col < rows_left ? (uint32_t)(r * ld + col) * 2u : kOob;
      } else {
        lk[it] = (pc ^ swz(r)) * 8;
        voff[it] = r < rows_left ? (uint32_t)(r * ld + lk[it]) * 2u : kOob;
      }
    }
  }
  // corner: the operand at the block's first row and the stage's first k, of which `left` are left to contract
  __device__ __forceinline__ void issue(const uint16_t* corner, EMI_LDS uint8_t* lds, int wave, int rows, int ld, int left) const {
    const uint32_t bytes = left <= 0 ? 0u : (uint32_t)(KM ? ((left < BK ? left : BK) - 1) * ld + rows : (rows - 1) * ld + left) * 2u;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(corner), 0, bytes, 0x00020000);
#pragma unroll
    for (int it = 0; it < LOADS; it++) {
      const uint32_t v = KM || lk[it] < left ? voff[it] : kOob;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, lds + (it * NW + wave) * 1024, 16, v, 0, 0, 0);
    }
  }
};

// WM x WN wavefronts tile the block's BM x BN; WK times as many share the k of every stage (k-step ks of 32 to the wavefronts
// ks % WK) and are added in wavefront order at the end.  A wavefront alone on its SIMD issues an instruction every 7 to 8 cycles,
// and a stage is forty for its loads and as many around its fragments and products: on few tiles that chain, and not the
// loads (64 bytes a cycle and CU, 258 cycles for 64 x 64 x 64), set the time.  Twice the wavefronts and stages twice as long, us, operands in the caches:
// 777 x 768 x 768 6.8 -> 5.5, x 2048 13.5 -> 9.0; 512 x 1024 x 1024 7.6 -> 6.0; 300 x 5632 x 2048 15.2 -> 13.2; 1000 x 2048 x 2048
// 14.5 -> 13.2; k-major B, three products summed: 777 x 768 x 768 14.8 -> 11.2.  part != nullptr: split-K, split z owns the stages
// [z * steps_per_split, ...) of the contraction (of the whole sum, where products are summed) and leaves its tile in
// part[z][M][N] for the reduction over splits.
// MODE: as in gemm_f32.hip; a lane has eight columns, four rotation pairs.  The product is rounded before the elementwise operator
// as it is when it goes through memory.  us, separate launches | together: gated 777 x 2048 x 768 21.8 | 14.0, 61 x 2048 x 768 7.2 | 6.5, 2181 x 1408 x
// 512 24.9 | 16.7; rotated 990 x 2048 x 2048 (three) 36.5 | 31.2, 777 x 768 x 768 12.2 | 9.3; adjoint 985 x 5632 x 2048 40.8 | 32.4,
// 777 x 2048 x 768 12.9 | 9.1.  Its other operand is read after the contraction: requested before, its registers cost the 128 x 128
// blocks more (990 x 2048 x 2048 49.6).
template <int MODE> struct PipeArg { using type = PipeSingle; };
template <> struct PipeArg<kTailGroup> { using type = PipeGroup; };
template <> struct PipeArg<kTailGated> {
  struct type {
    const uint16_t* B1;
    uint16_t *C1, *G;
  };
};
template <> struct PipeArg<kTailRotated> {
  struct type {
    const uint16_t* B[3];
    uint16_t* C[3];
    const float2* table;
    int seq, head_dim, rotated, pairs;
    const uint16_t *A1, *B1[3];
  };
};
template <> struct PipeArg<kTailAdjoint> {
  struct type {
    const uint16_t *h1, *h3;
    uint16_t* d3;
  };
};
__device__ __forceinline__ void unpack8(const u32x4_t r, float (&v)[8]) {
#pragma unroll
  for (int q = 0; q < 4; q++) {
    v[2 * q] = __uint_as_float(r[q] << 16);
    v[2 * q + 1] = __uint_as_float(r[q] & 0xffff0000u);
  }
}
__device__ __forceinline__ u32x4_t pack8(const float (&v)[8]) {
  return u32x4_t{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7])};
}

template <int BM, int BN, int WM, int WN, int WK, int BK, int NST, bool BKM, int MODE>
__global__ __launch_bounds__(WM* WN* WK * 64) void gemm_bf16_pipe_kernel(const uint16_t* A, const uint16_t* B, const uint16_t* R,
                                                                         uint16_t* C, int M, int N, int K, int lda, int ldb, int64_t ldr,
                                                                         int64_t ldc, int vec_ok, float* part, int steps_per_split,
                                                                         typename PipeArg<MODE>::type grp) {
  constexpr bool GROUPED = MODE == kTailGroup;
  constexpr int NW = WM * WN * WK;
  constexpr int TM = BM / WM / 16, TN = BN / WN / 16;
  constexpr int KS = BK / 32 / WK;                                // k-steps of 32 per wavefront and stage
  static_assert(NST >= 2 && KS >= 1 && BK == 32 * WK * KS, "stages");
  using OA = PipeOperand<BM, BK, NW, false>;
  using OB = PipeOperand<BN, BK, NW, BKM>;
  constexpr int STAGE = OA::BYTES + OB::BYTES;
  constexpr int LPT = OA::LOADS + OB::LOADS;
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem_raw[];
  EMI_LDS uint8_t* smem = (EMI_LDS uint8_t*)smem_raw;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l15 = lane & 15, g = lane >> 4;
  const int wk = wave / (WM * WN), wm = wave % (WM * WN) / WN, wn = wave % WN;

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
  const int64_t a_row = (int64_t)m0 * lda, b_row = BKM ? n0 : (int64_t)n0 * ldb;
  const int64_t b_k = BKM ? ldb : 1;                               // elements per k

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
    oa.issue(A + a_row + at_k, s, wave, rows_a, lda, left);
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

  f32x4_t acc[TM][TN];
#pragma unroll
  for (int a = 0; a < TM; a++)
#pragma unroll
    for (int b = 0; b < TN; b++)
#pragma unroll
      for (int r = 0; r < 4; r++) acc[a][b][r] = 0.f;

  // fragment of v_mfma_f32_16x16x32_bf16: lane l holds row l % 16, k = 8 (l / 16) .. + 7 of the k-step.  k-contiguous:
  // one 16-byte read of piece 4 ks + l / 16.  k-major: two transposing reads (k-rows 0..3 and 4..7 of the eight); within
  // 16 lanes, lane i addresses k-row i / 4, columns 4 (i % 4) .. + 3 and receives column i.
  [[maybe_unused]] uint32_t tr_at[TN];
  if constexpr (BKM) {
    const int kq = l15 >> 2;
#pragma unroll
    for (int b = 0; b < TN; b++) {
      const int col = wn * (BN / WN) + b * 16 + (l15 & 3) * 4, k = 32 * wk + 8 * g + kq;
      tr_at[b] = (uint32_t)(uintptr_t)smem + (uint32_t)(OA::BYTES + k * (BN * 2) + (((col >> 3) ^ OB::kswz(k)) << 4) + (col & 7) * 2);
    }
  }

#pragma unroll
  for (int s = 0; s < NST - 1; s++) issue();
  int slot = 0;
  auto contract = [&](int steps) __attribute__((always_inline)) {
  for (int t = 0; t < steps; t++) {
    pipe_wait_vmcnt<(NST - 2) * LPT>();                    // this stage has landed
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();                          // everyone's part of it, and the stage before is free again
    __builtin_amdgcn_sched_barrier(0);
    issue();
    const EMI_LDS uint8_t* sa = smem + slot * STAGE;
    const EMI_LDS uint8_t* sb = sa + OA::BYTES;
    const uint32_t stage_off = (uint32_t)(slot * STAGE);
    slot = slot + 1 < NST ? slot + 1 : 0;
    bf16x8_t fa[2][TM], fb[2][TN];
    auto read_kc = [&](const EMI_LDS uint8_t* base, int row, int ks) __attribute__((always_inline)) {
      return *reinterpret_cast<const EMI_LDS bf16x8_t*>(base + row * (BK * 2) + (((4 * ks + g) ^ OA::swz(row)) << 4));
    };
    auto read = [&](auto cc, bf16x8_t (&pa)[TM], bf16x8_t (&pb)[TN]) __attribute__((always_inline)) {
      constexpr int c = decltype(cc)::value;
      const int ks = c * WK + wk;
      if constexpr (BKM) {
        u32x2_t t[TN][2];
#pragma unroll
        for (int b = 0; b < TN; b++) {
          t[b][0] = pipe_tr_read<c * WK * 32 * BN * 2>(tr_at[b] + stage_off);
          t[b][1] = pipe_tr_read<(c * WK * 32 + 4) * BN * 2>(tr_at[b] + stage_off);
        }
#pragma unroll
        for (int a = 0; a < TM; a++) pa[a] = read_kc(sa, wm * (BM / WM) + a * 16 + l15, ks);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int b = 0; b < TN; b++) {
          asm volatile("" : "+v"(t[b][0]), "+v"(t[b][1]));          // not used, nor moved, before the wait
          const u32x4_t w = {t[b][0][0], t[b][0][1], t[b][1][0], t[b][1][1]};
          pb[b] = __builtin_bit_cast(bf16x8_t, w);
        }
      } else {
#pragma unroll
        for (int a = 0; a < TM; a++) pa[a] = read_kc(sa, wm * (BM / WM) + a * 16 + l15, ks);
#pragma unroll
        for (int b = 0; b < TN; b++) pb[b] = read_kc(sb, wn * (BN / WN) + b * 16 + l15, ks);
      }
    };
    auto multiply = [&](const bf16x8_t (&pa)[TM], const bf16x8_t (&pb)[TN]) __attribute__((always_inline)) {
      // operands swapped: a lane owns four consecutive columns
#pragma unroll
      for (int a = 0; a < TM; a++)
#pragma unroll
        for (int b = 0; b < TN; b++) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pb[b], pa[a], acc[a][b], 0, 0, 0);
    };
    read(std::integral_constant<int, 0>{}, fa[0], fb[0]);
    if constexpr (KS > 1) {
      static_assert(KS <= 2, "k-steps per stage");
      read(std::integral_constant<int, 1>{}, fa[1], fb[1]);
      __builtin_amdgcn_sched_barrier(0);
      multiply(fa[0], fb[0]);
      multiply(fa[1], fb[1]);
    } else {
      multiply(fa[0], fb[0]);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  };
  [[maybe_unused]] f32x4_t gate[TM][TN];                   // gated: the tile of h1
  if constexpr (MODE == kTailGated) {
    contract(ksteps);
#pragma unroll
    for (int a = 0; a < TM; a++)
#pragma unroll
      for (int b = 0; b < TN; b++) {
        gate[a][b] = acc[a][b];
        acc[a][b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
    contract(ksteps);
  } else {
    contract(nsteps);
  }
  pipe_wait_vmcnt<0>();                                    // the zero-filled loads past the end
  __syncthreads();

  // register r of lane l holds row l % 16, column 4 (l / 16) + r of its 16 x 16 tile.  Each wavefront lays its tile out
  // in the idle ring as fp32 rows; they are read back eight columns a lane, met by the residual and rounded once.
  constexpr int WR = BM / WM, WC = BN / WN, RS = WC + 4;
  EMI_LDS float* mine = (EMI_LDS float*)smem + wave * (WR * RS);
  auto lay = [&](const f32x4_t (&t)[TM][TN]) __attribute__((always_inline)) {
#pragma unroll
    for (int a = 0; a < TM; a++)
#pragma unroll
      for (int b = 0; b < TN; b++) *reinterpret_cast<EMI_LDS f32x4_t*>(mine + (a * 16 + l15) * RS + b * 16 + g * 4) = t[a][b];
    if constexpr (WK > 1) __syncthreads();
  };
  constexpr int PPR = WC / 8, PIECES = WR * PPR, THREADS = WK * 64, EACH = (PIECES + THREADS - 1) / THREADS;
  const int tile_wave = wave % (WM * WN), me = wk * 64 + lane;
  auto take = [&](int at, float (&v)[8]) __attribute__((always_inline)) {
    const int row = at / PPR, c8 = (at % PPR) * 8;
#pragma unroll
    for (int q = 0; q < 8; q++) v[q] = 0.f;
#pragma unroll
    for (int w = 0; w < WK; w++) {
      const EMI_LDS float* src = (EMI_LDS float*)smem + (w * WM * WN + tile_wave) * (WR * RS) + row * RS + c8;
      const f32x4_t lo = *reinterpret_cast<const EMI_LDS f32x4_t*>(src), hi = *reinterpret_cast<const EMI_LDS f32x4_t*>(src + 4);
#pragma unroll
      for (int q = 0; q < 4; q++) {
        v[q] += lo[q];
        v[4 + q] += hi[q];
      }
    }
  };
  [[maybe_unused]] u32x4_t h1[EACH];
  if constexpr (MODE == kTailGated) {
    lay(gate);
#pragma unroll
    for (int e = 0; e < EACH; e++) {
      const int at = e * THREADS + me;
      if (PIECES % THREADS != 0 && at >= PIECES) break;
      float v[8];
      take(at, v);
      h1[e] = pack8(v);
    }
    if constexpr (WK > 1) __syncthreads();
  }
  lay(acc);
#pragma unroll
  for (int e = 0; e < EACH; e++) {
    const int at = e * THREADS + me;
    if (PIECES % THREADS != 0 && at >= PIECES) break;
    const int row = at / PPR, c8 = (at % PPR) * 8;
    float v[8];
    take(at, v);
    const int grow = m0 + wm * WR + row, gcol = n0 + wn * WC + c8;
    if (grow >= M || gcol >= N) continue;
    if constexpr (MODE >= kTailGated) {                    // rows of whole pieces, results without a gap between them
      const int64_t to = (int64_t)grow * N + gcol;
      const u32x4_t y = pack8(v);
      if constexpr (MODE == kTailGated) {
        float a[8], o[8];
        unpack8(h1[e], a);
        unpack8(y, v);
#pragma unroll
        for (int q = 0; q < 8; q++) o[q] = emi_swiglu(a[q], v[q]);
        *reinterpret_cast<u32x4_t*>(C + to) = h1[e];
        *reinterpret_cast<u32x4_t*>(grp.C1 + to) = y;
        *reinterpret_cast<u32x4_t*>(grp.G + to) = pack8(o);
      } else if constexpr (MODE == kTailAdjoint) {
        float a[8], b[8], d1[8], d3[8];
        unpack8(*reinterpret_cast<const u32x4_t*>(grp.h1 + to), a);
        unpack8(*reinterpret_cast<const u32x4_t*>(grp.h3 + to), b);
        unpack8(y, v);
#pragma unroll
        for (int q = 0; q < 8; q++) emi_swiglu_adjoint(a[q], b[q], v[q], &d1[q], &d3[q]);
        *reinterpret_cast<u32x4_t*>(C + to) = pack8(d1);
        *reinterpret_cast<u32x4_t*>(grp.d3 + to) = pack8(d3);
      } else {
        u32x4_t z = y;
        if (outer < grp.rotated) {
          float o[8];
          unpack8(y, v);
          const float2* angles = grp.table + (int64_t)(grow % grp.seq) * (grp.head_dim >> 1);
#pragma unroll
          for (int q = 0; q < 4; q++) {
            const float2 t = angles[((gcol + 2 * q) % grp.head_dim) >> 1];
            o[2 * q] = rotated_even(t.x, t.y, v[2 * q], v[2 * q + 1]);
            o[2 * q + 1] = rotated_odd<bf16>(t.x, t.y, v[2 * q], v[2 * q + 1]);
          }
          z = pack8(o);
        }
        *reinterpret_cast<u32x4_t*>(C + to) = z;
      }
      continue;
    }
    if (part != nullptr) {
      float* dst = part + (int64_t)grow * N + gcol;
      if ((N & 3) == 0 && gcol + 8 <= N) {
        *reinterpret_cast<float4*>(dst) = make_float4(v[0], v[1], v[2], v[3]);
        *reinterpret_cast<float4*>(dst + 4) = make_float4(v[4], v[5], v[6], v[7]);
      } else {
#pragma unroll
        for (int q = 0; q < 8; q++)
          if (gcol + q < N) dst[q] = v[q];
      }
      continue;
    }
    uint16_t* dst = C + (int64_t)grow * ldc + gcol;
    const uint16_t* res = R != nullptr ? R + (int64_t)grow * ldr + gcol : nullptr;
    if (vec_ok && gcol + 8 <= N) {
      if (res != nullptr) {
        float r[8];
        unpack8(*reinterpret_cast<const u32x4_t*>(res), r);
#pragma unroll
        for (int q = 0; q < 8; q++) v[q] += r[q];
      }
      *reinterpret_cast<u32x4_t*>(dst) = pack8(v);
    } else {
#pragma unroll
      for (int q = 0; q < 8; q++)
        if (gcol + q < N) dst[q] = f32_to_bf16_bits(v[q] + (res != nullptr ? bf16_bits_to_f32(res[q]) : 0.f));
    }
  }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

int launch_bf16_splitk_reduce(hipStream_t st, const float* part, const uint16_t* R, uint16_t* C, int M, int N, int splits, int64_t ldr,
                              int64_t ldc);      // gemm.hip: adds `splits` planes [M, N] (+ R) into C in plane order

struct PipeCall {
  const uint16_t *A, *B, *R;
  uint16_t* C;
  int M, N, K, lda, ldb;
  int64_t ldr, ldc;
  int vec_ok;
  float* part;
  int splits;
  const PipeGroup* grp;       // nullptr: the single product of A and B
  int* planes;                // not null: splits stay planes in `part`, *planes of them (gemm_run)
};

// The ring of stages, and in the same place the wavefronts' tiles on their way out.
constexpr int pipe_lds(int bm, int bn, int wm, int wn, int wk, int bk, int nst) {
  const int ring = nst * (bm + bn) * bk * 2, tile = wm * wn * wk * (bm / wm) * (bn / wn + 4) * 4;
  return ring > tile ? ring : tile;
}

template <int BM, int BN, int WM, int WN, int WK, int BK, int NST, bool BKM, bool GROUPED>
static int launch_pipe_one(hipStream_t st, const PipeCall& c) {
  auto kern = gemm_bf16_pipe_kernel<BM, BN, WM, WN, WK, BK, NST, BKM, GROUPED ? kTailGroup : kTailNone>;
  constexpr int smem = pipe_lds(BM, BN, WM, WN, WK, BK, NST);
  static_assert(smem <= 160 * 1024, "LDS of a CU");
  static bool configured = false;
  if (const int rc = reserve_lds(reinterpret_cast<const void*>(kern), smem, configured)) return rc;
  const int steps = ((c.K + BK - 1) / BK) * (GROUPED && c.grp->sum ? c.grp->count : 1);
  const int sps = (steps + c.splits - 1) / c.splits, nz = (steps + sps - 1) / sps;
  const int outer = GROUPED && !c.grp->sum ? c.grp->count : nz;
  const int tiles = ((c.M + BM - 1) / BM) * ((c.N + BN - 1) / BN);
  float* part = outer == nz && nz > 1 ? c.part : nullptr;
  if constexpr (GROUPED)
    hipLaunchKernelGGL(kern, dim3(tiles * outer), dim3(WM * WN * WK * 64), smem, st, c.A, c.B, c.R, c.C, c.M, c.N, c.K, c.lda, c.ldb,
                       c.ldr, c.ldc, c.vec_ok, part, sps, *c.grp);
  else
    hipLaunchKernelGGL(kern, dim3(tiles * outer), dim3(WM * WN * WK * 64), smem, st, c.A, c.B, c.R, c.C, c.M, c.N, c.K, c.lda, c.ldb,
                       c.ldr, c.ldc, c.vec_ok, part, sps, PipeSingle{});
  EMI_CHECK_LAUNCH("emi_gemm");
  if (part != nullptr && c.planes != nullptr) {
    *c.planes = nz;
    return EMI_OK;
  }
  if (part != nullptr) return launch_bf16_splitk_reduce(st, part, c.R, c.C, c.M, c.N, nz, c.ldr, c.ldc);
  return EMI_OK;
}

template <int BM, int BN, int WM, int WN, int WK, int BK, int NST>
static int launch_pipe_shape(hipStream_t st, const PipeCall& c, int trans_b) {
  if (trans_b)
    return c.grp != nullptr ? launch_pipe_one<BM, BN, WM, WN, WK, BK, NST, false, true>(st, c)
                            : launch_pipe_one<BM, BN, WM, WN, WK, BK, NST, false, false>(st, c);
  if constexpr (BN >= 64)
    return c.grp != nullptr ? launch_pipe_one<BM, BN, WM, WN, WK, BK, NST, true, true>(st, c)
                            : launch_pipe_one<BM, BN, WM, WN, WK, BK, NST, true, false>(st, c);
  return -1;
}

// Which block and how many splits of K.  The estimate is of the CU with the most blocks, in microseconds: a start, the stages
// at the rate that each block shape was measured at with one, two, three and more blocks on the CU, the start of blocks that
// come after others, and what several results in one launch cost more.  Shape 0 is the 256 x 256 ping-pong kernel of gemm.hip,
// whose clock falls as it fills the chip, 1 the 128 x 128 tile of which two fit a CU, 2 the same tile in a ring of three stages
// whose k two wavefronts share, one to a CU, 3 128 x 64, 4 64 x 64, both in stages of 128 k, 5 a 32 x 32 tile whose eight
// wavefronts share stages of 256 k, 6 64 x 64 in stages of 64 k.  Fitted to products of 16 to 8192 tokens whose weights, 64 MB of
// them in turn, come from beyond the L2s, each with the blocks and splits that could be the fastest.  A k-major B has rates of
// its own, and with it 6 competes with 4: its stages hold a contraction of two or three of 128 k, or of splits so short, with
// less waste.  On 3991 other products the plan is 0.2 % (k-contiguous B) and 0.7 % (k-major; 2.1 % by the rates of the former)
// behind the fastest in the geometric mean.  us, B k-major, by those | these: 646 x 768 x 288 4.8 | 4.3, 18 x 288 x 288 x 3 summed
// 7.3 | 6.2, 32 x 768 x 2048 7.2 | 6.6, 344 x 768 x 2048 x 2 summed 14.6 | 12.3, 2499 x 1024 x 2816 30.5 | 24.5.
// The reduction over splits is a launch of its own; results over 4 M elements, whose planes leave the caches, are not split
// (but see pingpong_splits of gemm.hip), nor are the products of a few tokens, which have kernels of their own
// (gemm_skinny.hip).  A split of 64 x 64 tiles, and any with a k-major B, has at least three stages, others four.
Bf16Plan bf16_plan(int64_t M, int64_t N, int64_t K, int count, int sum, int trans_b, int64_t most) {
  struct Shape { int bm, bn, bk; double fixed, group, rate[3], more, later; };      // rate[b - 1]: per stage, b blocks on the CU; more: per
                                                                                   // block from four on; group: with several results; later:
                                                                                   // the start of each block that comes after others
  static const Shape shapes[6] = {
      {256, 256, 64, 4.0, 0.8, {1.0, 2.0, 3.0}, 1.0, 0.0},      {128, 128, 64, 3.9, 0.2, {0.59, 0.855, 1.6}, 0.515, 0.0},
      {128, 128, 64, 4.3, 0.3, {0.535, 1.07, 1.6}, 0.535, 0.0}, {128, 64, 128, 3.45, 0.45, {0.6, 1.24, 2.0}, 0.6, 0.0},
      {64, 64, 128, 3.15, 0.2, {0.355, 0.785, 1.10}, 0.41, 0.0}, {32, 32, 256, 3.4, 0.0, {0.30, 0.62, 1.4}, 0.363, 1.75}};
  static const Shape kmajor[7] = {
      {256, 256, 64, 4.0, 0.45, {1.0, 2.0, 3.0}, 1.0, 0.0},          {128, 128, 64, 5.1, 0.45, {0.585, 0.82, 1.435}, 0.50, 0.25},
      {128, 128, 64, 5.0, 0.45, {0.52, 1.05, 1.535}, 0.535, 3.35},    {128, 64, 128, 3.75, 0.45, {0.635, 1.20, 1.87}, 0.60, 0.5},
      {64, 64, 128, 3.0, 0.45, {0.415, 0.735, 1.29}, 0.41, 1.5},      {}, {64, 64, 64, 2.65, 0.45, {0.345, 0.43, 0.57}, 0.22, 0.9}};
  Bf16Plan best{1, 1, 0.0};
  double least = 1e30;
  const bool may_split = (sum || count == 1) && M * N <= (4 << 20) && M > 8 && K > 8;
  for (int c = 0; c < (trans_b ? 6 : 7); c++) {
    if ((c == 0 && sum && count > 1) || (c == 5 && !trans_b)) continue;        // what those kernels do not do
    const Shape& s = trans_b ? shapes[c] : kmajor[c];
    const int64_t steps = (K + s.bk - 1) / s.bk * (sum ? count : 1);
    const int64_t blocks = (M + s.bm - 1) / s.bm * ((N + s.bn - 1) / s.bn) * (sum ? 1 : count);
    if (blocks > 0x3fffffff) continue;
    const bool split = may_split && (c != 0 || trans_b);
    for (int64_t z = 1; z <= 16 && z <= most && (z == 1 || (split && steps >= (c == 4 || !trans_b ? 3 : 4) * z)); z++) {
      const int64_t b = (blocks * z + 255) / 256, per = (steps + z - 1) / z;
      double stage = b < 4 ? s.rate[b - 1] : s.more * b;
      const double later = c == 4 && trans_b ? (b > 2 ? 1.0 * (b - 2) : 0.0) : s.later * (b - 1);
      if (c == 0) stage *= 1.0 + 0.45 * (blocks * z < 256 ? blocks * z / 256.0 : 1.0);
      const double t = s.fixed + (count > 1 && !sum ? s.group : 0.0) + later + per * stage +
                       (z == 1 ? 0.0 : trans_b ? 2.8 + 0.78e-6 * M * N * (z + 1) : 2.65 + 1e-6 * M * N * (z + 1));
      if (t < least) {
        least = t;
        best = Bf16Plan{c, (int)z, t};
      }
    }
  }
  return best;
}

// The kernel of a plan's blocks: 0 the ping-pong kernel, 1, 2, 9 blocks of 128 x 128, 3, 4 of 128 x 64, 5 to 7 of 64 x 64, 8 of
// 32 x 32.
// More wavefronts and deeper rings, of stages of 128 k, where a block has its CU to itself and enough stages to fill them; 64 x 64
// blocks of four wavefronts and 64 k a stage, three of which fit a CU, where three there are, and of a k-major B where the
// plan says so or a contraction is of two or three stages.  us:
// 128 x 128, eight wavefronts | sixteen that share k: 1714 x 1408 x 512 8.4 | 8.7, 981 x 2816 x 1024 12.3 | 12.2, 520 x 4096 x 4096 36 | 33,
// 779 x 1408 x 512 (two) 9.1 | 9.8, 662 x 1024 x 1024 (three) 13.3 | 13.6, 3705 x 1024 x 1024 (three summed, B k-major) 30.6 | 31.3;
// 128 x 64, of 64 k and eight wavefronts | of 128 and sixteen: 512 x 768 x 768 (three) 9.1 | 8.4, 2048 x 768 x 288 5.5 | 6.2,
// 1000 x 1408 x 512 6.6 | 6.9, 3714 x 288 x 288 (three summed, B k-major) 9.7 | 10.1;
// 64 x 64, ring of two | three: 300 x 768 x 768 (B k-major) 6.7 | 6.1, 300 x 2816 x 1024 8.2 | 7.1, 256 x 2048 x 768 6.9 | 6.2,
// 300 x 1408 x 512 5.5 | 5.0, with B k-major 5.8 | 5.4, 493 x 512 x 512 4.7 | 4.9, 531 x 512 x 512 5.3 | 5.0;
// 64 x 64, of 128 | of 64 k: 1500 x 512 x 512 (three) 9.7 | 9.2, B k-major 270 x 768 x 288 4.6 | 4.4, 800 x 768 x 288 4.9 | 4.6.
int bf16_kernel(const Bf16Plan& plan, int64_t M, int64_t N, int64_t K, int count, int sum, int trans_b) {
  if (plan.shape == 2 && K < (count == 1 ? 1024 * plan.splits : sum ? 2560 : 2048)) return 9;
  if (plan.shape < 3) return plan.shape;
  if (plan.shape >= 5) return plan.shape == 5 ? 8 : 7;
  const int rows = plan.shape == 3 ? 128 : 64;
  const int64_t blocks = (M + rows - 1) / rows * ((N + 63) / 64) * (sum || count == 1 ? plan.splits : count), all_k = K * (sum ? count : 1);
  if (plan.shape == 3) return blocks <= 256 && all_k > 640 * plan.splits && K > 320 ? 4 : 3;
  if (blocks <= 256 && all_k >= (trans_b || N > 768 || blocks > 64 ? 512 : 640)) return 6;
  if (!trans_b) return all_k < 384 * plan.splits ? 7 : 5;
  return blocks > 512 && blocks <= 768 ? 7 : 5;
}

// C[i] = A[i] . op(B[i]) [+ R[i]] for i < count, or with `sum` the one sum of the products (+ R[0]), as the plan says
// (plan.shape >= 1; the caller has checked 16-byte rows).  vec_ok: 16-byte rows of C and R.
int launch_bf16_pipe(hipStream_t st, const Bf16Plan& plan, int count, const void* const* A, const void* const* B, const void* const* R,
                     void* const* C, float* part, int M, int N, int K, int lda, int ldb, int64_t ldr, int64_t ldc, int vec_ok, int trans_b,
                     int sum, int* planes) {
  PipeGroup g{};
  for (int i = 0; i < count; i++) {
    g.A[i] = static_cast<const uint16_t*>(A[i]);
    g.B[i] = static_cast<const uint16_t*>(B[i]);
  }
  for (int i = 0; i < (sum ? 1 : count); i++) {
    g.R[i] = R != nullptr ? static_cast<const uint16_t*>(R[i]) : nullptr;
    g.C[i] = static_cast<uint16_t*>(C[i]);
  }
  g.count = count;
  g.sum = sum;
  const PipeCall c{g.A[0], g.B[0], g.R[0], g.C[0], M, N, K, lda, ldb, ldr, ldc, vec_ok, part, part != nullptr ? plan.splits : 1,
                   count > 1 ? &g : nullptr, planes};
  switch (bf16_kernel(plan, M, N, K, count, sum, trans_b)) {
    case 1: return launch_pipe_shape<128, 128, 4, 2, 1, 64, 2>(st, c, trans_b);
    case 2: return launch_pipe_shape<128, 128, 4, 2, 2, 64, 3>(st, c, trans_b);
    case 3: return launch_pipe_shape<128, 64, 4, 2, 1, 64, 3>(st, c, trans_b);
    case 4: return launch_pipe_shape<128, 64, 4, 2, 2, 128, 3>(st, c, trans_b);
    case 5: return launch_pipe_shape<64, 64, 2, 2, 2, 128, 2>(st, c, trans_b);
    case 6: return launch_pipe_shape<64, 64, 2, 2, 2, 128, 3>(st, c, trans_b);
    case 7: return launch_pipe_shape<64, 64, 2, 2, 1, 64, 3>(st, c, trans_b);
    case 9: return launch_pipe_shape<128, 128, 4, 2, 1, 64, 3>(st, c, trans_b);
    default: return launch_pipe_shape<32, 32, 1, 1, 8, 256, 3>(st, c, trans_b);
  }
}

// The products of gemm_plan.h whose result goes through an elementwise operator.
template <int BM, int BN, int WM, int WN, int WK, int BK, int NST, bool BKM, int MODE>
static int launch_pipe_tail_one(hipStream_t st, const uint16_t* A, const uint16_t* B, const ProductTail& t, int M, int N, int K, int ldb) {
  auto kern = gemm_bf16_pipe_kernel<BM, BN, WM, WN, WK, BK, NST, BKM, MODE>;
  constexpr int smem = pipe_lds(BM, BN, WM, WN, WK, BK, NST);
  static bool configured = false;
  if (const int rc = reserve_lds(reinterpret_cast<const void*>(kern), smem, configured)) return rc;
  typename PipeArg<MODE>::type arg{};
  if constexpr (MODE == kTailGated) {
    arg = {static_cast<const uint16_t*>(t.B[1]), static_cast<uint16_t*>(t.C[1]), static_cast<uint16_t*>(t.C[2])};
  } else if constexpr (MODE == kTailRotated) {
    for (int i = 0; i < t.count; i++) {
      arg.B[i] = static_cast<const uint16_t*>(t.B[i]);
      arg.C[i] = static_cast<uint16_t*>(t.C[i]);
      arg.B1[i] = static_cast<const uint16_t*>(t.B1[i]);
    }
    arg.A1 = static_cast<const uint16_t*>(t.A1);
    arg.pairs = t.A1 != nullptr ? 2 : 1;
    arg.table = reinterpret_cast<const float2*>(t.table);
    arg.seq = t.seq, arg.head_dim = t.head_dim, arg.rotated = t.rotated;
  } else {
    arg = {static_cast<const uint16_t*>(t.h1), static_cast<const uint16_t*>(t.h3), static_cast<uint16_t*>(t.C[1])};
  }
  const int tiles = ((M + BM - 1) / BM) * ((N + BN - 1) / BN) * (MODE == kTailRotated ? t.count : 1);
  hipLaunchKernelGGL(kern, dim3(tiles), dim3(WM * WN * WK * 64), smem, st, A, B, (const uint16_t*)nullptr, static_cast<uint16_t*>(t.C[0]), M, N, K,
                     K, ldb, (int64_t)0, (int64_t)N, 1, (float*)nullptr, 0, arg);
  EMI_CHECK_LAUNCH("emi_gemm(elementwise tail)");
  return EMI_OK;
}
template <int BM, int BN, int WM, int WN, int WK, int BK, int NST>
static int launch_pipe_tail_shape(hipStream_t st, const uint16_t* A, const uint16_t* B, const ProductTail& t, int M, int N, int K, int ldb, int trans_b) {
  if (t.mode == kTailGated) return launch_pipe_tail_one<BM, BN, WM, WN, WK, BK, NST, false, kTailGated>(st, A, B, t, M, N, K, ldb);
  if (t.mode == kTailRotated) return launch_pipe_tail_one<BM, BN, WM, WN, WK, BK, NST, false, kTailRotated>(st, A, B, t, M, N, K, ldb);
  if (trans_b) return launch_pipe_tail_one<BM, BN, WM, WN, WK, BK, NST, false, kTailAdjoint>(st, A, B, t, M, N, K, ldb);
  if constexpr (BN >= 64) return launch_pipe_tail_one<BM, BN, WM, WN, WK, BK, NST, true, kTailAdjoint>(st, A, B, t, M, N, K, ldb);
  return -1;
}

// Against the separate launches by the plan's own estimates, and a pass of 2.4 us and the bytes it moves; a gated tile leaves
// three results, 1.2 to 2.2 us.  Over 135 products of 32 to 5000 rows by 768 x 288 to 5632 x 2048: 1.22 to 1.33 times as fast
// as the separate launches, none slower by more than 2 %.  What is for the 256-tiles goes there.
int launch_bf16_pipe_tail(hipStream_t st, const void* A, const void* B, const ProductTail& t, int M, int N, int K, int ldb, int trans_b) {
  if (t.mode != kTailAdjoint && !trans_b) return -1;
  const int count = t.mode == kTailGated ? 2 : t.mode == kTailRotated ? t.count : 1, sum = t.mode == kTailGated, pairs = t.A1 != nullptr ? 2 : 1;
  const Bf16Plan p = bf16_plan(M, N, (int64_t)K * pairs, count, sum, trans_b, 1), group = bf16_plan(M, N, K, count, 0, trans_b, 1),
                 one = bf16_plan(M, N, K, 1, 0, trans_b, kAnySplits);
  double apart = count * (one.us + 1.0) - 1.0;
  if (pairs == 2) {                                        // each result a launch that sums its two products, or two
    const double summed = bf16_plan(M, N, K, 2, 1, trans_b, sum_splits(M, N, kAnySplits)).us;
    apart = count * ((summed < 2 * one.us + 1.0 ? summed : 2 * one.us + 1.0) + 1.0) - 1.0;
  } else if (group.us < apart) {
    apart = group.us;
  }
  const double moved = 2e-6 / 5.0 * M * N * (t.mode == kTailRotated ? 2 * t.rotated : t.mode == kTailGated ? 3 : 5);
  const double pass = t.mode == kTailRotated && t.rotated == 0 ? 0.0 : 2.4 + moved;
  const double results = t.mode != kTailGated ? 0.0 : p.shape == 5 ? 1.2 : 2.2;
  if (p.shape == 0 || (one.shape == 0 && pairs == 1) || p.us + results >= apart + pass) return -1;
  const uint16_t *a = static_cast<const uint16_t*>(A), *b = static_cast<const uint16_t*>(B);
  switch (bf16_kernel(p, M, N, (int64_t)K * pairs, count, sum, trans_b)) {
    case 1: return launch_pipe_tail_shape<128, 128, 4, 2, 1, 64, 2>(st, a, b, t, M, N, K, ldb, trans_b);
    case 2: return launch_pipe_tail_shape<128, 128, 4, 2, 2, 64, 3>(st, a, b, t, M, N, K, ldb, trans_b);
    case 3: return launch_pipe_tail_shape<128, 64, 4, 2, 1, 64, 3>(st, a, b, t, M, N, K, ldb, trans_b);
    case 4: return launch_pipe_tail_shape<128, 64, 4, 2, 2, 128, 3>(st, a, b, t, M, N, K, ldb, trans_b);
    case 5: return launch_pipe_tail_shape<64, 64, 2, 2, 2, 128, 2>(st, a, b, t, M, N, K, ldb, trans_b);
    case 6: return launch_pipe_tail_shape<64, 64, 2, 2, 2, 128, 3>(st, a, b, t, M, N, K, ldb, trans_b);
    case 7: return launch_pipe_tail_shape<64, 64, 2, 2, 1, 64, 3>(st, a, b, t, M, N, K, ldb, trans_b);
    case 9: return launch_pipe_tail_shape<128, 128, 4, 2, 1, 64, 3>(st, a, b, t, M, N, K, ldb, trans_b);
    default: return launch_pipe_tail_shape<32, 32, 1, 1, 8, 256, 3>(st, a, b, t, M, N, K, ldb, trans_b);
  }
}

}  // namespace emi
