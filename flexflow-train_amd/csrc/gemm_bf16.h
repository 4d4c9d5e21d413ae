// The bf16 MFMA kernels behind gemm.hip, and the rules that choose among them.  A template of the
// transposes that gemm_nn.hip, gemm_nt.hip, gemm_tn.hip, gemm_tt.hip and gemm_tail_*.hip instantiate
// (the kernels take minutes to compile; these files compile side by side).
#pragma once
#include "lds_dma.h"
#include "gemm.h"
#include "colreduce.h"
#include "gemm_any.h"
#include <algorithm>
#include <stdarg.h>
#include <stdio.h>
#include <string.h>
#include <type_traits>
#include <utility>

namespace ffk {

__device__ __forceinline__ float apply_activation(float v, int act) {
  switch (act) {
    case FFK_ACT_RELU:
      // tensor_accessor_relu keeps x >= 0 (tensor_accessor_unary_ops.cc:32-38);
      // identical to x > 0 ? x : 0 on every input except -0.0f.
      return v >= 0.0f ? v : 0.0f;
    case FFK_ACT_SIGMOID:
      return 1.0f / (1.0f + expf(-v));
    case FFK_ACT_TANH:
      return tanhf(v);
    case FFK_ACT_GELU:
      return gelu_forward(v);
    default:
      return v;
  }
}

// ---------------------------------------------------------------------------
// Block -> tile mapping.  Workgroups are dealt round-robin to the 8 XCDs, each
// with its own L2; regroup ids so that one XCD works on a compact patch of the
// output (tiles that share A rows / B columns), then walk the patch in groups
// of kGroupM tile rows.  (xcds: how many of them share these tiles.)
// ---------------------------------------------------------------------------
__device__ __forceinline__ void tile_coords(int pid, int nbm, int nbn, int &tm,
                                            int &tn, int xcds = kNumXCD) {
  int const total = nbm * nbn;
  {
    // XCD x gets a contiguous run of total / 8 tiles, the first total % 8 of them one more
    int const xcd = pid % xcds;
    int const local = pid / xcds;
    pid = xcd * (total / xcds) + min(xcd, total % xcds) + local;
  }
  constexpr int kGroupM = 8;
  int const group_size = kGroupM * nbn;
  int const group = pid / group_size;
  int const first_m = group * kGroupM;
  int const rows = min(nbm - first_m, kGroupM);
  int const in_group = pid % group_size;
  tm = first_m + in_group % rows;
  tn = in_group / rows;
}

// ---------------------------------------------------------------------------
// Asking instead of launching: while this thread's name sink is set (by
// ffk_gemm_kernel_name), every launch site below adds the kernel it would
// have launched to the sink and returns without touching the device.
// ---------------------------------------------------------------------------
inline thread_local char *tl_name_sink = nullptr;
inline thread_local size_t tl_name_sink_bytes = 0;
inline bool describe_only(char const *fmt, ...) __attribute__((format(printf, 1, 2)));
inline bool describe_only(char const *fmt, ...) {
  if (tl_name_sink == nullptr) return false;
  size_t used = strlen(tl_name_sink);
  if (used > 0 && used + 4 < tl_name_sink_bytes) used += strlen(strcpy(tl_name_sink + used, " + "));
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(tl_name_sink + used, tl_name_sink_bytes - used, fmt, ap);
  va_end(ap);
  return true;
}
inline char const *tf(bool b) { return b ? "true" : "false"; }

// ---------------------------------------------------------------------------
// bf16 MFMA kernel
// ---------------------------------------------------------------------------
// eight / the first few bytes of a row at any address
struct __attribute__((packed, aligned(2))) Raw8 { u32x2 v; };
__device__ __forceinline__ u32x2 load_any8(bf16 const *p) { return reinterpret_cast<Raw8 const *>(p)->v; }
__device__ __forceinline__ u32x2 load_first4(bf16 const *p, int n) {
  u32x4 const v = load_raw_first(p, n);
  return u32x2{v[0], v[1]};
}

// f of 0, 1, ..., as constants (a loop of this many long bodies is not unrolled)
template <int... I, typename F>
__device__ __forceinline__ void unroll_for(std::integer_sequence<int, I...>, F f) {
  (f(std::integral_constant<int, I>{}), ...);
}

// acc += a . b with the accumulator in accumulation registers.  Written as an instruction: of 256 accumulator and 128
// fragment registers the compiler keeps some of each kind in the other kind's place, and then moves 108 of them
// there and back in every k-tile ([16384, 4096] . [12288, 4096]^T 1473 us, 1194 so).  It does not see
// that these results take time: mfma16_settled has to stand between the last of them and their first use.
__device__ __forceinline__ void mfma16_in_place(f32x4 &acc, bf16x8 a, bf16x8 b) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}
// ... and a direct load behind it: the MFMA stands between the write of M0 and the load that reads it, where lds_dma16 has
// a wait state.  (The descriptor needs more of them: uniform_pointer in lds_dma.h.)
__device__ __forceinline__ void mfma16_in_place_and_load(f32x4 &acc, bf16x8 a, bf16x8 b, i32x4 rsrc, unsigned lane_byte_off,
                                                         unsigned uniform_byte_off, unsigned lds_byte_addr) {
  asm volatile("s_mov_b32 m0, %3\n\tv_mfma_f32_16x16x32_bf16 %0, %1, %2, %0\n\tbuffer_load_dwordx4 %4, %5, %6 offen lds"
               : "+a"(acc)
               : "v"(a), "v"(b), "s"(lds_byte_addr), "v"(lane_byte_off), "s"(rsrc), "s"(uniform_byte_off)
               : "memory");
}
template <int N>
__device__ __forceinline__ void mfma16_settled(f32x4 (&acc)[N]) {
#pragma unroll
  for (int i = 0; i < N; i++) asm volatile("s_nop 7" : "+a"(acc[i]));
}

enum { kEdgeNone = 0, kEdgeOverlap = 1, kEdgeBounded = 2 };

// The register-staged kernel: operands at any address with any row stride (the tile and what it costs are
// in gemm_any.h).
template <int BM, int BN, int WM, int WN, bool TA, bool TB>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * 64) void gemm_bf16_kernel(
    bf16 const *__restrict__ A, bf16 const *__restrict__ B, bf16 *C, int M,
    int N, int K, int64_t lda, int64_t ldb, int64_t ldc,
    bf16 const *__restrict__ bias, int act, int accumulate) {
  using Tile = AnyTile<BM, BN, WM, WN, !TA, TB>;
  __shared__ __attribute__((aligned(16))) bf16 smem[2 * Tile::kBufElems];
  int tm, tn;
  tile_coords(blockIdx.x, (M + BM - 1) / BM, (N + BN - 1) / BN, tm, tn);
  int const m0 = tm * BM, n0 = tn * BN;
  typename Tile::OpA a;
  typename Tile::OpB b;
  a.init(A, nullptr, lda, M, K, 0, m0, threadIdx.x);
  b.init(B, nullptr, ldb, N, K, 0, n0, threadIdx.x);
  Tile tile;
  tile.template reduce<false>(a, b, K, 0, (K + kBK - 1) / kBK, smem);
  tile.store(m0, n0, M, N, [&](int m, int n, float v) {
    if (bias != nullptr) v += VecIO<bf16>::load1(bias + n);
    v = apply_activation(v, act);
    bf16 *const dst = C + (int64_t)m * ldc + n;
    if (accumulate) v += VecIO<bf16>::load1(dst);
    VecIO<bf16>::store1(dst, v);
  });
}

// ---------------------------------------------------------------------------
// bf16 MFMA kernel, pipelined: shapes that tile exactly, and with EDGE also tiles
// that begin early (kEdgeOverlap) or guard their edges (kEdgeBounded):
//  * operand tiles go global -> LDS directly (global_load_lds_dwordx4, no VGPR
//    staging, no LDS write instructions) into a ring of STAGES buffers, so the
//    loads of the next STAGES-1 k-tiles are in flight while one is consumed --
//    this is what hides HBM/L2 latency when only one workgroup fits a CU;
//  * a direct load writes 64 lanes x 16 B contiguously, so bank conflicts are
//    avoided by permuting which 16-byte chunk each lane FETCHES (an XOR
//    swizzle) instead of padding rows;
//  * the accumulator tile is computed transposed (B as the first MFMA operand)
//    so that a lane holds 4 consecutive output columns, staged through LDS and
//    written to HBM as full 16-byte chunks with bias/activation/accumulate
//    applied on the way.
// ---------------------------------------------------------------------------
// PF = how many k-steps ahead of its use a fragment is read from LDS (PF + 1
// register buffers).  3 on the 64x64 tiles, whose waves have one MFMA per k-step;
// 1 on the larger ones: on the 128x128 tile (2 MFMAs per k-step per wave) 3
// gained nothing.
// Column sums add up blocks of 32 rows as four runs of 8 (colsum_partial_vec_kernel below).
constexpr int kColsumRowsPerLane = 8;
constexpr int kColsumRowsPerBlock = 4 * kColsumRowsPerLane;

struct GemmTailArgs {
  bf16 const *in;
  bf16 *out;
  DropoutParams dropout;
  // kTailDropout*Grad only, optional: [M / 32][N] sums of 32-row blocks of
  // what the tail stores, added up in colsum_partial_vec_kernel's order
  float *colsum_partials;
};

// Further GEMMs of the same kind and reduction length run by the same launch: workgroups from
// first_tile of a problem on compute it.
struct GemmGroupArgs {
  struct Problem {
    bf16 const *A, *B;
    bf16 *C;
    int64_t lda, ldb, ldc;
    int M, N;
    int first_tile;  // number of tiles (= workgroups) of the problems before it
  } p[kMaxGemmGroup - 1];
  int count;  // of p
  // Column reductions that ride along: workgroups from first_sum on.  They read what earlier launches left, and
  // run where the tiles leave CUs idle; a launch of their own is 3 to 7 us of latency (encoder layers forward and
  // backward, batch x tokens x width: 8 x 512 x 1024 511 -> 504 us, 7 x 197 x 768 247.5 -> 242, 2 x 48 x 128 69 -> 67
  // replayed from a graph, within noise launched one by one).
  int first_sum;
  ColreduceBatch sums;
};
struct GemmNoGroup {};

// TAIL (GemmEpilogue::Tail): element-wise operators applied to the 8-element
// pieces of the output tile on their way from LDS to memory.
// GROUP: the launch carries several problems (no bias, no split-K).
// EDGE: M, N and K need not be whole tiles (the operands still have to be readable 16 bytes at a
// time).  Two ways:
//   kEdgeOverlap (M >= BM, N >= BN): the last row and column of tiles begin early enough to lie inside
//     the output, and do not store what their neighbours store.  No load needs a bound but those of a
//     ragged last k-tile, whose lanes past K ask for an offset past the descriptor's bound and get
//     zeros; the steady loop stops one tile earlier and is that of whole tiles.
//   kEdgeBounded (any M, N): lanes whose rows or columns lie past the operand ask for an offset past the
//     descriptor's bound and get zeros, for which each load of a K-contiguous panel keeps lane offsets of
//     its own.  (A descriptor per load, bounded by what is left of the operand, took 20% of the loop of a
//     128x128 tile, 4095 x 1024 over 4096: 39.0 us, 32.6 with 4096 rows, and 8% of a 64x64 one.)
// KG: groups of waves that each take a part of the reduction (with LDS stages of their own) and add
// up their accumulators at the end.  A 64x64 tile is 4 MFMAs a wave and k-tile, which a barrier, an
// LDS round trip and the MFMAs' own dependence stretch to some 600 cycles; a second group fills them
// where there are too few tiles for a second workgroup per CU.
// With four groups of one wave a 32x32 tile, no barrier stands in the loop.  Where the tiles leave CUs idle,
// a workgroup's time is the bytes it reads over what its LDS stages can have in flight for the some 800 ns
// they take to come: a quarter of the tile reads half the bytes and there are four times the workgroups
// (405 x 512 over 2048 8.8 -> 6.3 us, 63 x 768 over 3072 10.2 -> 6.7, 756 x 256 over 768 5.5 -> 4.5), and the
// output's operators are spread over all of its waves (96 x 256 over 128 with GELU and dropout 7.3 -> 5.3).
template <int BM, int BN, int WM, int WN, int BK, int STAGES, int PF, bool TA, bool TB, int TAIL = 0,
          bool GROUP = false, int EDGE = kEdgeNone, int KG = 1>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * 64 * KG) void gemm_bf16_pipe_kernel(
    bf16 const *__restrict__ A, bf16 const *__restrict__ B, bf16 *C, int M,
    int N, int K, int64_t lda, int64_t ldb, int64_t ldc,
    bf16 const *__restrict__ bias, int act, int accumulate,
    float *__restrict__ partial, int k_tiles_per_split, GemmTailArgs tail, std::conditional_t<GROUP, GemmGroupArgs, GemmNoGroup> group) {
  extern __shared__ __attribute__((aligned(16))) bf16 smem[];
  int bid = blockIdx.x;
  if constexpr (GROUP) {
    int const id = bid;
    if (id >= group.first_sum) {
      colreduce_batch_block<bf16, (BM / WM) * (BN / WN) * 64 * KG>(group.sums, id - group.first_sum,
                                                                   *reinterpret_cast<float (*)[32][33]>(smem));
      return;
    }
#pragma unroll
    for (int q = 0; q < kMaxGemmGroup - 1; q++) {
      if (q < group.count && id >= group.p[q].first_tile) {  // uniform over the workgroup
        bid = id - group.p[q].first_tile;
        A = group.p[q].A, B = group.p[q].B, C = group.p[q].C;
        M = group.p[q].M, N = group.p[q].N;
        lda = group.p[q].lda, ldb = group.p[q].ldb, ldc = group.p[q].ldc;
      }
    }
  }
  // partial != nullptr: split-K.  Workgroup (tile, split) reduces k-tiles
  // [split * k_tiles_per_split, +k_tiles_per_split) and stores its fp32
  // accumulators to partial[split][M][N]; a second kernel sums the splits and
  // applies the epilogue.
  constexpr int NW = (BM / WM) * (BN / WN);
  constexpr int NT = NW * 64;
  // a group is one wave: nobody but the wave itself reads its stages, and no barrier stands in its loop
  constexpr bool ALONE = NW == 1 && KG > 1;
  // One wave per SIMD and two stages: see the k-loop.
  constexpr bool WIDE2 = WM == 128 && (WN == 128 || WN == 96) && STAGES == 2;
  // M16: on v_mfma_f32_16x16x32_bf16 instead of v_mfma_f32_32x32x16_bf16: the same bits (measured over reductions of 32
  // to 4096) for less power.  With operands in registers alone, all CUs busy and normally distributed values, the
  // first runs at 2.04 PFLOP/s and the second at 1.80, both at the clock that power leaves them.
  // (The wide tile, launch to launch, and with what the k-loop says of the order of its loads: [16384, 4096] . [12288,
  // 4096]^T 1242 -> 1143 us, [16384, 12288] . [12288, 4096] 1320 -> 1214, [12288, 16384] . [16384, 4096] with A transposed
  // 1271 -> 1215, [4096, 1024] . [4096, 1024]^T 40 -> 36-37.)
  constexpr bool M16 = WIDE2;
  constexpr int MB = M16 ? 16 : 32, MK = M16 ? 32 : 16;  // rows and columns, and k's, of a matrix instruction
  using Acc = std::conditional_t<M16, f32x4, f32x16>;
  constexpr int TM = WM / MB, TN = WN / MB;
  constexpr bool TBL = (TB == false);  // B tile lies as [BK][BN]
  constexpr int A_ELEMS = BM * BK, B_ELEMS = BN * BK;
  constexpr int A_LOADS = A_ELEMS / 8 / NT, B_LOADS = B_ELEMS / 8 / NT;
  constexpr int LPT = A_LOADS + B_LOADS;  // direct loads per thread per k-tile
  constexpr int STAGE_ELEMS = A_ELEMS + B_ELEMS;
  constexpr int CPRK = BK / 8;             // 16-byte chunks per K-contiguous row
  constexpr int RPW = 256 / (BK * 2);      // K-contiguous rows per 256-byte bank window
  constexpr int CS = WN + 8;               // row stride of a wave's staged output tile
  static_assert(A_ELEMS / 8 % NT == 0 && B_ELEMS / 8 % NT == 0, "tile/threads");
  static_assert(STAGES * LPT <= 63, "vmcnt range");

  static_assert(KG == 1 || EDGE == kEdgeBounded, "written for this");
  int const kg = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / NT);
  int const t = KG == 1 ? threadIdx.x : threadIdx.x % NT, lane = t & 63, wave = t >> 6;
  int const wm0 = (wave / (BN / WN)) * WM;
  int const wn0 = (wave % (BN / WN)) * WN;
  int tm, tn;
  int const nbm = EDGE ? (M + BM - 1) / BM : M / BM, nbn = EDGE ? (N + BN - 1) / BN : N / BN;
  int const tiles = nbm * nbn;
  int split = 0;
  if (partial == nullptr) {
    tile_coords(bid, nbm, nbn, tm, tn);
  } else {
    // an XCD's workgroups take the same split: its part of the operands then passes through that
    // L2 alone
    int const splits = gridDim.x / tiles;
    split = bid % splits;
    tile_coords(bid / splits, nbm, nbn, tm, tn, splits < kNumXCD ? kNumXCD / splits : 1);
  }
  // (kEdgeOverlap) what of the tile is this workgroup's to store begins at first_m, first_n
  int const first_m = tm * BM, first_n = tn * BN;
  // (an operand whose contiguous index is M may be padded to whole 16-byte chunks: rows past M are
  // loaded then, and not stored)
  int const M_loads = TA && EDGE ? (M + 7) & ~7 : M;
  int const m0 = EDGE == kEdgeOverlap ? min(first_m, M_loads - BM) : first_m, n0 = EDGE == kEdgeOverlap ? min(first_n, N - BN) : first_n;
  // first k-tile of this workgroup, or of this group of waves
  int const kt0 = KG == 1 ? split * k_tiles_per_split : kg * (((K + BK - 1) / BK + KG - 1) / KG);

  // Per-lane offset of its first chunk inside the block's operand panel; the
  // chunk of load i lies a uniform number of rows further on, and the k-tile
  // advances a uniform base, so a load address is a scalar base plus one
  // 32-bit lane offset that never changes.
  // K-contiguous tile [rows][BK]: physical chunk pc of a row holds logical
  // chunk pc ^ ((row / RPW) % CPRK).  Tile lying as [BK][cols]: the 64-byte
  // segment s of row k sits at segment s ^ (k % 4) (with 64 columns, whose rows are
  // half a bank window, at s ^ ((k / 2) % 2); with 32 there is one).
  // For M16, whose transposing reads take rows k and k + 8 side by side, 32 bytes of each: the 32-byte piece p of row k
  // sits at p ^ (2 (k % 4) + (k / 8) % 2).
  auto tr_swizzle = [](int krow, int cols) { return cols == 32 ? 0 : cols == 64 ? (krow >> 1) & 1 : krow & 3; };
  auto tr_chunk = [&](int krow, int pc, int cols) {  // the 16-byte chunk of the row that lies at chunk pc
    return M16 ? pc ^ ((((krow & 3) << 1) | ((krow >> 3) & 1)) << 1) : (((pc >> 2) ^ tr_swizzle(krow, cols)) << 2) | (pc & 3);
  };
  constexpr int ROWS_PER_LOAD_KC = NT / CPRK;     // rows covered by one load of all threads
  static_assert((ROWS_PER_LOAD_KC / RPW) % CPRK == 0, "swizzle must repeat per load");
  static_assert((!TA || (NT * 8 % BM == 0 && (NT * 8 / BM) % 4 == 0)) && (!TBL || (NT * 8 % BN == 0 && (NT * 8 / BN) % 4 == 0)),
                "a panel lying [BK][cols] must divide into whole loads, and the swizzle repeat per load");
  unsigned voff_a, voff_b;
  {
    int c = wave * 64 + lane;
    if (!TA) {
      int row = c / CPRK, pc = c % CPRK;
      int lc = pc ^ ((row / RPW) & (CPRK - 1));
      voff_a = (unsigned)(row * lda + lc * 8) * 2u;
    } else {
      constexpr int CPR = BM / 8;
      int krow = c / CPR, pc = c % CPR;
      int lc = tr_chunk(krow, pc, BM);
      voff_a = (unsigned)(krow * lda + lc * 8) * 2u;
    }
    if (!TBL) {
      int row = c / CPRK, pc = c % CPRK;
      int lc = pc ^ ((row / RPW) & (CPRK - 1));
      voff_b = (unsigned)(row * ldb + lc * 8) * 2u;
    } else {
      constexpr int CPR = BN / 8;
      int krow = c / CPR, pc = c % CPR;
      int lc = tr_chunk(krow, pc, BN);
      voff_b = (unsigned)(krow * ldb + lc * 8) * 2u;
    }
  }
  int const KT_all = EDGE ? (K + BK - 1) / BK : K / BK;  // k-tiles of the whole reduction
  int64_t const step_a = TA ? (int64_t)(NT * 8 / BM) * lda : (int64_t)ROWS_PER_LOAD_KC * lda;
  int64_t const step_b = TBL ? (int64_t)(NT * 8 / BN) * ldb : (int64_t)ROWS_PER_LOAD_KC * ldb;
  bf16 const *const panel_a = uniform_pointer(TA ? A + m0 : A + (int64_t)m0 * lda);
  bf16 const *const panel_b = uniform_pointer(TBL ? B + n0 : B + (int64_t)n0 * ldb);
  // (kEdgeBounded) lanes whose rows or columns lie past the operand ask for what no descriptor covers and get
  // zeros: of a K-contiguous panel each load has rows of its own, of one lying [BK][cols] all have the lane's columns
  constexpr bool ROWS_A = EDGE == kEdgeBounded && !TA, ROWS_B = EDGE == kEdgeBounded && !TBL;
  // (M16) loads of 8 rows of a panel lying [BK][cols] take turns between two offsets, 32 bytes apart
  constexpr bool TURN_A = M16 && TA && NT * 8 / BM == 8, TURN_B = M16 && TBL && NT * 8 / BN == 8;
  static_assert(!M16 || (EDGE != kEdgeBounded && (!TA || TURN_A || NT * 8 / BM % 16 == 0) && (!TBL || TURN_B || NT * 8 / BN % 16 == 0)),
                "written for these loads");
  unsigned off_a[ROWS_A ? A_LOADS : TURN_A ? 2 : 1], off_b[ROWS_B ? B_LOADS : TURN_B ? 2 : 1];
  {
    int const c = wave * 64 + lane;
    auto columns_from = [&](int cols) {  // of the lane's pieces (see the swizzle above)
      int const krow = c / (cols / 8), pc = c % (cols / 8);
      return (((pc >> 2) ^ tr_swizzle(krow, cols)) << 5) | ((pc & 3) << 3);
    };
#pragma unroll
    for (int q = 0; q < (ROWS_A ? A_LOADS : 1); q++) {
      bool const there = EDGE != kEdgeBounded || (TA ? m0 + columns_from(BM) < M_loads : m0 + c / CPRK + q * ROWS_PER_LOAD_KC < M);
      off_a[q] = there ? voff_a : 0x80000000u;
    }
#pragma unroll
    for (int q = 0; q < (ROWS_B ? B_LOADS : 1); q++) {
      bool const there = EDGE != kEdgeBounded || (TBL ? n0 + columns_from(BN) < N : n0 + c / CPRK + q * ROWS_PER_LOAD_KC < N);
      off_b[q] = there ? voff_b : 0x80000000u;
    }
  }
  if constexpr (TURN_A) {
    int const c = wave * 64 + lane;
    off_a[1] = (unsigned)(c / (BM / 8) * lda + tr_chunk(c / (BM / 8) + 8, c % (BM / 8), BM) * 8) * 2u;
  }
  if constexpr (TURN_B) {
    int const c = wave * 64 + lane;
    off_b[1] = (unsigned)(c / (BN / 8) * ldb + tr_chunk(c / (BN / 8) + 8, c % (BN / 8), BN) * 8) * 2u;
  }
  auto lane_a = [&](int q) __attribute__((always_inline)) { return off_a[ROWS_A ? q : TURN_A ? q & 1 : 0]; };
  auto lane_b = [&](int q) __attribute__((always_inline)) { return off_b[ROWS_B ? q : TURN_B ? q & 1 : 0]; };

  // WIDE2: a ring of five panels, A's and B's of the k-tiles in turn (see the k-loop); `stage` is where a tile's A lies.
  constexpr int RING = 5, PANEL = A_ELEMS > B_ELEMS ? A_ELEMS : B_ELEMS;
  auto ring_at = [](int at, int d) __attribute__((always_inline)) { return at + d >= RING ? at + d - RING : at + d; };
  // LDS destinations of the direct loads are scalar byte addresses: base + stage + chunk row
  bf16 *const stages = smem + (KG == 1 ? 0 : kg * (STAGES * STAGE_ELEMS));
  unsigned const smem_addr = lds_address_of(stages);
  int const wave_s = __builtin_amdgcn_readfirstlane(wave);
  // Loads [first, first + count) of a k-tile's LPT direct loads (A's, then B's).
  // (first and count are constants once the caller's loops are unrolled)
  // (maybe_last: the k-tile may be the last one of the reduction)
  auto issue_some = [&](int kt, int stage, int first, int count, bool maybe_last) __attribute__((always_inline)) {
    unsigned const sa = smem_addr + (unsigned)(WIDE2 ? stage * PANEL : stage * STAGE_ELEMS) * 2u;
    unsigned const sb = WIDE2 ? smem_addr + (unsigned)(ring_at(stage, 1) * PANEL) * 2u : sa + (unsigned)A_ELEMS * 2u;
    unsigned const bound = EDGE == kEdgeBounded ? 0x80000000u : 0xffffffffu;
    if constexpr (EDGE != kEdgeNone) {
      if (maybe_last && kt0 + kt >= KT_all - 1 && (K % BK != 0 || kt0 + kt >= KT_all)) {  // uniform over the wave
        i32x4 const ra = buffer_resource(panel_a + (TA ? (int64_t)(kt0 + kt) * BK * lda : (int64_t)(kt0 + kt) * BK), 0x80000000u);
        i32x4 const rb = buffer_resource(panel_b + (TBL ? (int64_t)(kt0 + kt) * BK * ldb : (int64_t)(kt0 + kt) * BK), 0x80000000u);
        // k's of this tile, none for a group of waves that ran out of k-tiles
        int const left = kt0 + kt >= KT_all ? 0 : K - (KT_all - 1) * BK;
        int const c = wave * 64 + lane;
        bool const past = ((c % CPRK) ^ ((c / CPRK / RPW) & (CPRK - 1))) * 8 >= left;  // this lane's k's of a K-contiguous panel
#pragma unroll
        for (int q = 0; q < LPT; q++) {
          if (q < first || q >= first + count) continue;
          if (q < A_LOADS) {
            bool const there = !TA ? !past : c / (BM / 8) + q * (NT * 8 / BM) < left;
            lds_dma16(ra, there ? lane_a(q) : 0x80000000u, (unsigned)(q * step_a) * 2u, sa + (unsigned)(q * NW + wave_s) * 1024u);
          } else {
            int const i = q - A_LOADS;
            bool const there = !TBL ? !past : c / (BN / 8) + i * (NT * 8 / BN) < left;
            lds_dma16(rb, there ? lane_b(i) : 0x80000000u, (unsigned)(i * step_b) * 2u, sb + (unsigned)(i * NW + wave_s) * 1024u);
          }
        }
        return;
      }
    }
    i32x4 const ra = buffer_resource(panel_a + (TA ? (int64_t)(kt0 + kt) * BK * lda : (int64_t)(kt0 + kt) * BK), bound);
    i32x4 const rb = buffer_resource(panel_b + (TBL ? (int64_t)(kt0 + kt) * BK * ldb : (int64_t)(kt0 + kt) * BK), bound);
#pragma unroll
    for (int q = 0; q < LPT; q++) {
      if (q < first || q >= first + count) continue;
      if (q < A_LOADS) {
        lds_dma16(ra, lane_a(q), (unsigned)(q * step_a) * 2u, sa + (unsigned)(q * NW + wave_s) * 1024u);
      } else {
        int const i = q - A_LOADS;
        lds_dma16(rb, lane_b(i), (unsigned)(i * step_b) * 2u, sb + (unsigned)(i * NW + wave_s) * 1024u);
      }
    }
  };
  // (WIDE2) f(descriptor, lane offset, uniform offset, LDS address) of load q of a k-tile that is not the last one;
  // panel: where in the ring what it is part of goes
  auto load_operands = [&](int kt, int panel, int q, auto f) __attribute__((always_inline)) {
    static_assert(EDGE != kEdgeBounded || !M16, "no bound in the descriptor");
    if (q < A_LOADS) {
      f(buffer_resource(panel_a + (TA ? (int64_t)(kt0 + kt) * BK * lda : (int64_t)(kt0 + kt) * BK)), lane_a(q),
        (unsigned)(q * step_a) * 2u, smem_addr + (unsigned)(panel * PANEL) * 2u + (unsigned)(q * NW + wave_s) * 1024u);
    } else {
      int const i = q - A_LOADS;
      f(buffer_resource(panel_b + (TBL ? (int64_t)(kt0 + kt) * BK * ldb : (int64_t)(kt0 + kt) * BK)), lane_b(i),
        (unsigned)(i * step_b) * 2u, smem_addr + (unsigned)(panel * PANEL) * 2u + (unsigned)(i * NW + wave_s) * 1024u);
    }
  };
  auto issue = [&](int kt, int stage) {
    issue_some(kt, stage, 0, LPT, true);
  };

  // Fragment readers (see the layouts above).  Everything lane-dependent in
  // an LDS address is tabulated once here; inside the loop an address is
  // stage base + table entry + a compile-time constant that folds into the
  // instruction's offset field, so the k-loop carries almost no address math.
  constexpr int KS = BK / MK;  // MFMA k-steps per tile
  // K-contiguous tile: lane l reads row (row0 + l%32), logical chunk 2 kk + l/32 (M16: l%16, 4 kk + l/16).
  // row0 is a multiple of 32 (16), so the swizzle term depends on the lane only.
  int kc_off[KS];
  {
    int const sw = ((lane & (MB - 1)) / RPW) & (CPRK - 1);
    static_assert(!M16 || 16 / RPW % CPRK == 0, "the swizzle repeats every 16 rows");
#pragma unroll
    for (int kk = 0; kk < KS; kk++) {
      kc_off[kk] = (lane & (MB - 1)) * BK + (((MK / 8 * kk + lane / MB) ^ sw) << 3);
    }
  }
  auto frag_kc = [&](bf16 const *tile, int row0, int kk) -> bf16x8 {
    return *reinterpret_cast<bf16x8 const *>(tile + kc_off[kk] + row0 * BK);
  };
  // Tile lying as [BK][cols]: lane reads rows kk*16 + 8 (l/32) + (l%16)/4 (+4),
  // columns col0 + 16 ((l/16)%2) + 4 (l%4); the 64-byte segment index is
  // XOR-ed with tr_swizzle(row), which touches only its two low bits (its one bit).
  // One entry per 32-wide block of the wave's tile.  M16: rows kk*32 + 8 (l/16) + (l%16)/4 (+4), columns
  // col0 + 4 (l%4), one entry per 16-wide block.
  int tr_tab_a[TM], tr_tab_b[TN];
  if constexpr (M16) {
    int const krow = (lane >> 4) * 8 + ((lane & 15) >> 2);
    auto offset = [&](int cols, int block) {
      return krow * cols + ((block ^ (((krow & 3) << 1) | ((krow >> 3) & 1))) << 4) + (lane & 3) * 4;
    };
#pragma unroll
    for (int i = 0; i < TM; i++) tr_tab_a[i] = offset(BM, (wm0 >> 4) + i);
#pragma unroll
    for (int j = 0; j < TN; j++) tr_tab_b[j] = offset(BN, (wn0 >> 4) + j);
  } else {
    int const i16 = lane & 15;
    int const q = i16 >> 2;
    int const inseg = ((lane >> 4) & 1) * 16 + (i16 & 3) * 4;
    int const krow = (lane >> 5) * 8 + q;
    auto offset = [&](int cols, int block) {
      return krow * cols + (((block & 3) ^ tr_swizzle(q, cols)) << 5) + ((block & ~3) << 5) + inseg;
    };
#pragma unroll
    for (int i = 0; i < TM; i++) tr_tab_a[i] = offset(BM, (wm0 >> 5) + i);
#pragma unroll
    for (int j = 0; j < TN; j++) tr_tab_b[j] = offset(BN, (wn0 >> 5) + j);
  }
  auto frag_tr = [&](bf16 const *tile, int rowlen, int tab, int kk) -> bf16x8 {
    bf16 const *p = tile + tab + kk * MK * rowlen;
    typedef s16x4 __attribute__((address_space(3))) * lds_s16x4_ptr;
    s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(p));
    s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(p + 4 * rowlen));
    union {
      s16x4 h[2];
      bf16x8 v;
    } u;
    u.h[0] = lo;
    u.h[1] = hi;
    return u.v;
  };

  Acc acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int r = 0; r < (M16 ? 4 : 16); r++) acc[i][j][r] = 0.0f;

  int const KT = KG > 1 ? (KT_all + KG - 1) / KG : partial != nullptr ? (EDGE ? min(k_tiles_per_split, KT_all - kt0) : k_tiles_per_split) : KT_all;
  constexpr int NB = PF + 1;  // fragment buffers
  static_assert(KS % NB == 0, "buffer index must not depend on the tile");
  static_assert(STAGES >= 2, "one stage in use, at least one in flight");
  // With three or more stages a refill is not issued in one burst after the
  // barrier that frees its stage, but in KS equal parts: part 0 after that
  // barrier, part j in k-step j-1 of the following tile.  A burst of LPT loads
  // from every wave at once overruns the memory pipeline's instruction queue;
  // a wave that cannot issue its next load cannot issue its next MFMA either.
  constexpr bool SPREAD = STAGES >= 3 && LPT % KS == 0;
  constexpr int PART = SPREAD ? LPT / KS : LPT;
  // (One wave per SIMD and two stages: a refill goes out behind the barrier that frees its stage.)
  constexpr int PRO_PART = WIDE2 ? LPT : PART;  // of the last tile the prologue starts
#pragma unroll
  for (int s = 0; s < STAGES; s++) {
    if (s < KT) {
      if (SPREAD && s == STAGES - 1) {
        issue_some(s, s, 0, PRO_PART, true);  // tile 0's steps issue the rest
      } else {
        issue(s, WIDE2 ? 2 * s : s);
      }
    }
  }
  // Fragments are double-buffered in registers: while the MFMAs of one k-step
  // run, the LDS reads of the next step (of the next tile, at a tile's last
  // step) are already in flight.
  bf16x8 af[NB][TM], bfr[NB][TN];
  auto read_frags = [&](int buf, int stage, int kk) {
    bf16 const *sa = stages + stage * STAGE_ELEMS;
    bf16 const *sb = sa + A_ELEMS;
#pragma unroll
    for (int i = 0; i < TM; i++) {
      af[buf][i] = TA ? frag_tr(sa, BM, tr_tab_a[i], kk) : frag_kc(sa, wm0 + i * 32, kk);
    }
#pragma unroll
    for (int j = 0; j < TN; j++) {
      bfr[buf][j] = TBL ? frag_tr(sb, BN, tr_tab_b[j], kk) : frag_kc(sb, wn0 + j * 32, kk);
    }
  };
  // (M16, one wave per SIMD) one fragment of k-step kk of the panel at `at` in the ring
  auto read_a16 = [&](int at, int i, int kk) __attribute__((always_inline)) {
    bf16 const *sa = smem + at * PANEL;
    af[kk][i] = TA ? frag_tr(sa, BM, tr_tab_a[i], kk) : frag_kc(sa, wm0 + i * 16, kk);
  };
  auto read_b16 = [&](int at, int j, int kk) __attribute__((always_inline)) {
    bf16 const *sb = smem + at * PANEL;
    bfr[kk][j] = TBL ? frag_tr(sb, BN, tr_tab_b[j], kk) : frag_kc(sb, wn0 + j * 16, kk);
  };
  constexpr int EARLY = 3;  // A's fragments of a tile's first step that are read before it begins
  // Tile 0 must have landed (STAGES-1 younger tiles may still be in flight).
  if (STAGES - 1 < KT) {
    wait_vmcnt<(STAGES - 2) * LPT + PRO_PART>();
  } else {
    wait_vmcnt<0>();
  }
  // Barrier without a memory fence: a fence would wait for every direct load
  // still in flight; the vmcnt waits already cover the tile that is needed.
  if constexpr (!ALONE) asm volatile("s_barrier" ::: "memory");
  if constexpr (M16) {
#pragma unroll
    for (int j = 0; j < TN; j++) read_b16(1, j, 0);
#pragma unroll
    for (int i = 0; i < EARLY; i++) read_a16(0, i, 0);
  } else {
#pragma unroll
    for (int kk = 0; kk < PF; kk++) read_frags(kk, 0, kk);
  }
  // One k-tile.  STEADY: every condition of the generic body is known true
  // (next tile exists, a refill is due, STAGES-2 younger tiles in flight), so
  // the steady-state loop is branch-free.
  // SST: the tile's stage when the caller knows it (the steady loop, unrolled by STAGES), -1
  // otherwise.  With the stage a constant every LDS address of the tile is a loop-invariant
  // register plus an immediate; computed from kt it costs three vector instructions per k-step,
  // which two waves on a SIMD do not get for free.
  [[maybe_unused]] int ring = 0;  // (WIDE2) where the tile's A lies
  auto tile_step = [&](int kt, auto steady_tag, auto stage_tag) __attribute__((always_inline)) {
    constexpr bool STEADY = decltype(steady_tag)::value;
    constexpr int SST = decltype(stage_tag)::value;
    auto stage_at = [&](int d) { return SST >= 0 ? (SST + d) % STAGES : (kt + d) % STAGES; };
    int const stage = stage_at(0);
    if constexpr (WIDE2) {
      // One wave per SIMD: nothing but this wave's own instruction order hides a latency, so
      // the order is written out.  A tile is two k-steps of TM * TN MFMAs, row block by row block; behind an MFMA
      // sits at most one fragment read or one direct load, fenced so that the compiler keeps them there.
      //   step 0   reads the rest of its own A fragments, each some 20 MFMAs ahead of its use, and all of step 1's;
      //            A's panel of the tile after the next goes out
      //   step 1   after BARRIER MFMAs every wave has what it needs of this tile, and the next one has landed: from
      //            there on the next tile's B fragments and the first of A's are read, and B's panel of the
      //            tile after it goes out
      // LDS holds five panels: this tile's two, the next one's, and A's of the one after that, which takes the place of B's of
      // the tile before.  So loads go out evenly over the whole tile (a CU takes in 64 bytes a cycle, 1024 of the
      // 2048 cycles; all of them behind the barrier, and the waves waited to get theirs in: [12288,
      // 16384] . [16384, 4096] with A transposed 1384 us, 1228 so) and have 85 MFMAs' time and more, 1360 cycles, to land.
      static_assert(PF == 1 && KS == 2 && TM == 8 && TN % 2 == 0, "written for these shapes");
      constexpr int NS = TM * TN, BARRIER = NS / 4;
      constexpr int R0 = TM - EARLY + TN + TM, R1 = TN + EARLY;  // reads of the two steps, in even slots; loads in odd ones
      static_assert(2 * R0 <= NS && 2 * R1 <= NS - BARRIER && 2 * A_LOADS <= NS && 2 * B_LOADS <= NS - BARRIER, "slots");
      bool const next = STEADY || kt + 1 < KT, after = STEADY || kt + 2 < KT;
      int const own_b = ring_at(ring, 1), next_a = ring_at(ring, 2), next_b = ring_at(ring, 3), after_a = ring_at(ring, 4);
      // step 0's read r: A3, B0, B1, A4, B2, B3, ... (A's of this step, B's of the next one), then the other B's and all A's of the next
      auto read0 = [&](int r) __attribute__((always_inline)) {
        constexpr int OWN = TM - EARLY;
        if (r < 2 * OWN) {
          if (r % 2 == 0) read_a16(ring, EARLY + r / 2, 0);
          else read_b16(own_b, r / 2, 1);
        } else if (r < OWN + TN) {
          read_b16(own_b, r - OWN, 1);
        } else {
          read_a16(ring, r - OWN - TN, 1);
        }
      };
      auto read1 = [&](int r) __attribute__((always_inline)) {
        if (r == 0 || r > TN) read_a16(next_a, r == 0 ? 0 : r - TN, 0);
        else read_b16(next_b, r - 1, 0);
      };
      // which of `count`, spread over every other slot from `first` on, sits behind MFMA m (-1: none)
      auto behind = [](int m, int first, int count) constexpr {
        for (int i = 0; i < count; i++) {
          if (first + 2 * (i * ((NS - first) / 2) / count) == m) return i;
        }
        return -1;
      };
      auto mfma = [&](auto kk_tag, auto m_tag) __attribute__((always_inline)) {
        constexpr int kk = decltype(kk_tag)::value, m = decltype(m_tag)::value;
        constexpr int r = behind(m, kk == 0 ? 0 : BARRIER, kk == 0 ? R0 : R1);
        constexpr int l = behind(m, kk == 0 ? 1 : BARRIER + 1, kk == 0 ? A_LOADS : B_LOADS);
        Acc &d = acc[m / TN][m % TN];
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (l >= 0 && STEADY) {
          load_operands(kt + 2, kk == 0 ? after_a : ring, kk == 0 ? l : A_LOADS + l,
                        [&](i32x4 rsrc, unsigned off, unsigned uniform, unsigned lds) __attribute__((always_inline)) {
            mfma16_in_place_and_load(d, bfr[kk][m % TN], af[kk][m / TN], rsrc, off, uniform, lds);
          });
        } else {
          mfma16_in_place(d, bfr[kk][m % TN], af[kk][m / TN]);
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (l >= 0 && !STEADY) {
          if (after) issue_some(kt + 2, after_a, kk == 0 ? l : A_LOADS + l, 1, true);
        }
        if constexpr (kk == 1 && m == BARRIER - 1) {
          if (next) {
            // younger than the next tile's panels is A's of the one after it
            if (after) wait_vmcnt<A_LOADS>();
            else wait_vmcnt<0>();
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
          }
        }
        if constexpr (r >= 0) {
          if constexpr (kk == 0) read0(r);
          else if (next) read1(r);
        }
      };
      unroll_for(std::make_integer_sequence<int, NS>{}, [&](auto m) __attribute__((always_inline)) { mfma(std::integral_constant<int, 0>{}, m); });
      unroll_for(std::make_integer_sequence<int, NS>{}, [&](auto m) __attribute__((always_inline)) { mfma(std::integral_constant<int, 1>{}, m); });
      __builtin_amdgcn_sched_barrier(0);
      ring = ring_at(ring, 2);
      return;
    }
    if constexpr (!WIDE2) {
#pragma unroll
    for (int kk = 0; kk < KS; kk++) {
      int const cur = kk % NB;
      int const nxt = (kk + PF) % NB;  // buffer of the step read now
      // The first MFMA of the step is issued before the prefetch below so that
      // the wait for this step's fragments does not also cover the reads
      // issued now (the hardware counter is in order).
      __builtin_amdgcn_sched_barrier(0);
      acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bfr[cur][0], af[cur][0], acc[0][0], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (SPREAD && kk + 1 < KS) {
        // part kk+1 of the tile that goes into the stage freed one tile ago
        if (STEADY || kt + STAGES - 1 < KT) {
          issue_some(kt + STAGES - 1, stage_at(STAGES - 1), (kk + 1) * PART, PART, !STEADY);
        }
      }
      if (kk + PF < KS) {
        read_frags(nxt, stage, kk + PF);
      } else if (STEADY || kt + 1 < KT) {
        if (kk + PF == KS) {
          // First read of tile kt+1: make it visible and refill this tile's own
          // stage -- under this step's MFMAs, which cover those latencies.
          // Every wave has all fragments of tile kt in registers once its LDS
          // counter drains, so after the barrier the stage is free.
          if (STEADY || kt + STAGES - 1 < KT) {
            // (PF = 3 reads the next tile one step before the last part of a refill goes out: of
            // what is younger than the next tile's own last part, two parts are missing)
            static_assert(!SPREAD || PF <= 2 || (PF == 3 && KS == 4), "count of younger loads");
            wait_vmcnt<(STAGES - 2) * LPT - (SPREAD && PF == 3 ? 2 * PART : 0)>();
          } else {
            wait_vmcnt<0>();
          }
          if constexpr (ALONE) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
          else asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
          if (STEADY || kt + STAGES < KT) {
            issue_some(kt + STAGES, stage, 0, PART, !STEADY);
          }
        }
        read_frags(nxt, stage_at(1), kk + PF - KS);
      }
      __builtin_amdgcn_sched_barrier(0);
      // Transposed accumulation: rows of the MFMA result = output columns.
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
          if (i + j > 0)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bfr[cur][j], af[cur][i], acc[i][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    }
  };
  using Dyn = std::integral_constant<int, -1>;
  int kt = 0;
  // the steady loop asks for no tile from here on (a group's own last k-tiles may lie past the others')
  int const KT_steady = EDGE != kEdgeNone ? KT - KG : KT;
  if constexpr (!WIDE2 && (STAGES == 4 || STAGES == 2)) {
    for (; kt + 2 * STAGES - 1 < KT_steady; kt += STAGES) {  // kt % STAGES == 0, all STAGES tiles steady
      tile_step(kt, std::true_type{}, std::integral_constant<int, 0>{});
      tile_step(kt + 1, std::true_type{}, std::integral_constant<int, 1>{});
      if constexpr (STAGES == 4) {
        tile_step(kt + 2, std::true_type{}, std::integral_constant<int, 2>{});
        tile_step(kt + 3, std::true_type{}, std::integral_constant<int, 3>{});
      }
    }
  }
  for (; kt + STAGES < KT_steady; kt++) {
    tile_step(kt, std::true_type{}, Dyn{});
  }
  for (; kt < KT; kt++) {
    tile_step(kt, std::false_type{}, Dyn{});
  }
  // acc[i][j][r]: output row m = wm0 + 32 i + lane % 32,
  //               column n = wn0 + 32 j + 8 (r / 4) + 4 (lane / 32) + r % 4;
  // M16:          row m = wm0 + 16 i + lane % 16, column n = wn0 + 16 j + 4 (lane / 16) + r.
  // Both are groups of four consecutive columns (GROUPS to a block).
  constexpr int GROUPS = M16 ? 1 : 4;
  if constexpr (M16) mfma16_settled(acc[TM - 1]);
  auto row_of = [&](int i) __attribute__((always_inline)) { return i * MB + (lane & (MB - 1)); };
  auto col_of = [&](int j, int g) __attribute__((always_inline)) { return j * MB + 8 * g + 4 * (lane / MB); };
  // The plain store (no tail, nothing to add to): straight from the registers.  A lane holds four columns of a
  // block; swapping every other row of 16 lanes between a pair of blocks gives each lane 8 columns of one of the two,
  // so that every lane stores 16 bytes and four lanes together 64 contiguous bytes of a row.  No LDS, so no barrier either:
  // a wave writes its tile as soon as its own loop is done.  Used by the one-wave-per-SIMD kernel, where it
  // was 4-6% of a launch at reductions up to 2048; with two waves per SIMD the staged
  // epilogue below, whose stores are whole 128-byte lines, is 2-5% ahead.
  // Eight columns from column n of row m on (EDGE: those that exist).
  auto store8 = [&](int m, int n, u32x4 v) __attribute__((always_inline)) {
    bf16 *const to = C + (int64_t)m * ldc + n;
    if constexpr (EDGE == kEdgeOverlap) {
      if (m < first_m || n + 8 <= first_n || (TA && m >= M)) return;
      store_raw_any(to, v);
    } else if constexpr (EDGE == kEdgeBounded) {
      if (m >= M || n >= N) return;
      if (n + 8 <= N) {
        store_raw_any(to, v);
      } else {
        store_raw_first(to, v, N - n);
      }
    } else {
      *reinterpret_cast<u32x4 *>(to) = v;
    }
  };
  // Bias of four columns from n on.
  auto bias4 = [&](int n, float (&bv)[4]) __attribute__((always_inline)) {
    if constexpr (EDGE == kEdgeBounded) {
#pragma unroll
      for (int e = 0; e < 4; e++) bv[e] = bias != nullptr && n + e < N ? VecIO<bf16>::load1(bias + n + e) : 0.0f;
    } else {
      u32x2 raw = {0u, 0u};
      if (bias != nullptr) raw = EDGE != kEdgeNone ? load_any8(bias + n) : *reinterpret_cast<u32x2 const *>(bias + n);
      bv[0] = __uint_as_float(raw[0] << 16);
      bv[1] = __uint_as_float(raw[0] & 0xffff0000u);
      bv[2] = __uint_as_float(raw[1] << 16);
      bv[3] = __uint_as_float(raw[1] & 0xffff0000u);
    }
  };
  if constexpr (TAIL == GemmEpilogue::kTailNone && WIDE2) {
    if (partial == nullptr && accumulate == 0) {  // uniform over the launch
      auto direct = [&](auto actf) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < TN; j += 2) {
          float bv[2][4];
#pragma unroll
          for (int jj = 0; jj < 2; jj++) bias4(n0 + wn0 + col_of(j + jj, 0), bv[jj]);
          int const h = lane >> 4, n = (j + (h & 1)) * 16 + (h >> 1) * 8;
#pragma unroll
          for (int i = 0; i < TM; i++) {
            uint32_t w[2][2];
#pragma unroll
            for (int jj = 0; jj < 2; jj++) {
              float v[4];
#pragma unroll
              for (int e = 0; e < 4; e++) v[e] = actf(acc[i][j + jj][e] + bv[jj][e]);
              w[jj][0] = pack_bf16x2(v[0], v[1]);
              w[jj][1] = pack_bf16x2(v[2], v[3]);
            }
            // swaps the odd rows of 16 lanes of the first operand with the even rows of the second
            auto const lo = __builtin_amdgcn_permlane16_swap(w[0][0], w[1][0], false, false);
            auto const hi = __builtin_amdgcn_permlane16_swap(w[0][1], w[1][1], false, false);
            u32x4 const out = {lo[0], hi[0], lo[1], hi[1]};
            store8(m0 + wm0 + row_of(i), n0 + wn0 + n, out);
          }
        }
      };
      direct([](float v) { return v; });  // (this kernel is only launched without an activation)
      return;
    }
  }
  // Column sums of a staged tile of `rows` x `cols` from row m, column n on.  A thread owns a column; per block of
  // 32 rows: four runs of 8 rows summed in row order, then (0 + 1) + (2 + 3).
  auto column_sums = [&](bf16 const *staged, int stride, int rows, int cols, int m, int n, int first, int threads) __attribute__((always_inline)) {
    for (int i = first; i < cols * (rows / kColsumRowsPerBlock); i += threads) {
      int const col = i % cols, blk = i / cols;
      float run[4];
#pragma unroll
      for (int q = 0; q < 4; q++) {
        float acc_rows = 0.0f;
#pragma unroll
        for (int r = 0; r < kColsumRowsPerLane; r++) {
          acc_rows += VecIO<bf16>::load1(staged + (blk * kColsumRowsPerBlock + q * kColsumRowsPerLane + r) * stride + col);
        }
        run[q] = acc_rows;
      }
      int64_t const part = m / kColsumRowsPerBlock + blk;
      if (EDGE == kEdgeBounded && (part * kColsumRowsPerBlock >= M || n + col >= N)) continue;
      tail.colsum_partials[part * N + n + col] = (run[0] + run[1]) + (run[2] + run[3]);
    }
  };
  constexpr bool kColsums = TAIL == GemmEpilogue::kTailDropoutGeluGrad || TAIL == GemmEpilogue::kTailDropoutReluGrad;
  static_assert(!kColsums || EDGE != kEdgeOverlap, "blocks of 32 rows begin at multiples of 32");
  // Eight results from column n of row m on, rounded, to memory through the tail's operators.  kept: the
  // piece's place in the staged tile.
  auto put_piece = [&](int m, int n, u32x4 v, bf16 *kept) __attribute__((always_inline)) {
    int64_t const at = (int64_t)m * ldc + n;
    if constexpr (TAIL == GemmEpilogue::kTailNone) {
      store8(m, n, v);
    } else {
      if constexpr (EDGE == kEdgeOverlap) {  // N is a multiple of 8 here: a piece is one workgroup's
        if (m < first_m || n < first_n) return;
      }
      if constexpr (EDGE == kEdgeBounded) {  // ... or not there
        if (m >= M || n >= N) {
          *reinterpret_cast<u32x4 *>(kept) = u32x4{0u, 0u, 0u, 0u};  // for the column sums
          return;
        }
      }
      // ldc == N here: `at` is the element's index in the dense tensor, and
      // the piece is one block of the dropout stream
      uint32_t w[4] = {0u, 0u, 0u, 0u};
      // At a rate of zero everything is kept, whatever the stream says.  Only the residual add of a
      // backward (always rate zero) asks: the branch keeps the pieces' loads from running under one
      // another (forward of 4096 x 4096 -> 1024 with dropout and add: 45 us with it, 42 without).
      if (!(TAIL == GemmEpilogue::kTailDropoutAdd && !TB) || tail.dropout.threshold != 0) {
        philox4x32_10((tail.dropout.offset + (uint64_t)at) >> 3, tail.dropout.key, w);
      }
      u32x4 aux = {0u, 0u, 0u, 0u};
      if constexpr (TAIL == GemmEpilogue::kTailGeluDropout || TAIL == GemmEpilogue::kTailActDropout) {
        *reinterpret_cast<u32x4 *>(C + at) = v;
      } else {
        aux = *reinterpret_cast<u32x4 const *>(tail.in + at);
      }
      u32x4 r;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        float x[2] = {__uint_as_float(v[q] << 16), __uint_as_float(v[q] & 0xffff0000u)};
        float const a[2] = {__uint_as_float(aux[q] << 16), __uint_as_float(aux[q] & 0xffff0000u)};
#pragma unroll
        for (int h = 0; h < 2; h++) {
          if constexpr (TAIL == GemmEpilogue::kTailGeluDropout) {
            x[h] = storage_round<bf16>(gelu_forward(x[h]));
          }
          x[h] = keep(w, 2 * q + h, tail.dropout) ? x[h] * tail.dropout.scale : 0.0f;
          if constexpr (TAIL == GemmEpilogue::kTailDropoutGeluGrad) {
            x[h] = storage_round<bf16>(x[h]) * gelu_derivative(a[h]);
          }
          if constexpr (TAIL == GemmEpilogue::kTailDropoutReluGrad) {
            x[h] = a[h] > 0.0f ? x[h] : 0.0f;
          }
          if constexpr (TAIL == GemmEpilogue::kTailDropoutAdd) {
            x[h] = storage_round<bf16>(x[h]) + a[h];
          }
        }
        r[q] = pack_bf16x2(x[0], x[1]);
      }
      bf16 *const to = TAIL == GemmEpilogue::kTailGeluDropout || TAIL == GemmEpilogue::kTailActDropout ? tail.out : C;
      *reinterpret_cast<u32x4 *>(to + at) = r;
      if constexpr (kColsums) {
        // kept for the column sums below (the lane's own piece: no other lane reads it before the barrier)
        if (tail.colsum_partials != nullptr) *reinterpret_cast<u32x4 *>(kept) = r;
      }
    }
  };
  if constexpr (ALONE) {
    // Every wave lays down its sums in its own stages, 16 bytes a lane and access (66 lanes' room for each 64:
    // what eight lanes read side by side below then lies in different banks); then all threads add up pieces
    // of eight columns over the waves, in their order, and finish them.
    static_assert(TM * TN * 4 * 66 * 8 <= STAGES * STAGE_ELEMS, "a tile's sums fit a wave's stages");
    f32x4 *const mine = reinterpret_cast<f32x4 *>(stages) + lane;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
          mine[((i * TN + j) * 4 + g) * 66] = f32x4{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
        }
    __syncthreads();
    constexpr int AS = BN + 8;
    bf16 *const tile_kept = smem + KG * (STAGES * STAGE_ELEMS);
    auto pieces = [&](auto actf) __attribute__((always_inline)) {
      for (int c = threadIdx.x; c < BM * BN / 8; c += KG * 64) {
        int const row = c / (BN / 8), ch = c % (BN / 8), m = m0 + row, n = n0 + ch * 8;
        int const at = (((row >> 5) * TN + (ch >> 2)) * 4 + (ch & 3)) * 66 + (row & 31);
        f32x4 lo = {0.0f, 0.0f, 0.0f, 0.0f}, hi = lo;
#pragma unroll
        for (int o = 0; o < KG; o++) {
          f32x4 const *const part = reinterpret_cast<f32x4 const *>(smem + o * (STAGES * STAGE_ELEMS)) + at;
          lo += part[0];
          hi += part[32];
        }
        float v[8], old[8];
        float bv[2][4];
        bias4(n, bv[0]);
        bias4(n + 4, bv[1]);
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = actf((e < 4 ? lo[e & 3] : hi[e & 3]) + bv[e >> 2][e & 3]);
        if (accumulate != 0 && m < M && n < N) {
          // add the old value in fp32 before the single rounding
          bf16 const *const from = C + (int64_t)m * ldc + n;
          unpack_raw(n + 8 <= N ? load_raw_any(from) : load_raw_first(from, N - n), old, (bf16 const *)nullptr);
#pragma unroll
          for (int e = 0; e < 8; e++) v[e] += old[e];
        }
        put_piece(m, n, pack_raw(v, (bf16 const *)nullptr), tile_kept + row * AS + ch * 8);
      }
    };
    if (act == FFK_ACT_NONE) {
      pieces([](float v) { return v; });
    } else if (act == FFK_ACT_GELU) {
      pieces([](float v) { return gelu_forward(v); });
    } else if (act == FFK_ACT_RELU) {
      pieces([](float v) { return v >= 0.0f ? v : 0.0f; });
    } else {
      pieces([act](float v) { return apply_activation(v, act); });
    }
    if constexpr (kColsums) {
      if (tail.colsum_partials != nullptr) {  // uniform over the launch
        __syncthreads();
        column_sums(tile_kept, AS, BM, BN, m0, n0, (int)threadIdx.x, KG * 64);
      }
    }
    return;
  }
  __syncthreads();  // all stages are free now: reuse them for the output tile
  if constexpr (KG > 1 && !ALONE) {
    static_assert((KG - 1) * NW * TM * TN * 1024 <= (KG - 1) * STAGES * STAGE_ELEMS / 2, "partial tiles fit the groups' stages");
    // group g's accumulators, 16 bytes a lane and access, in the stages that were group g's (the
    // output tile is staged in group 0's)
    f32x4 *const mine = reinterpret_cast<f32x4 *>(stages) + wave * (TM * TN * 4 * 64) + lane;
    if (kg > 0) {
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
          for (int g = 0; g < 4; g++) {
            mine[((i * TN + j) * 4 + g) * 64] =
                f32x4{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
          }
    }
    __syncthreads();
    if (kg > 0) return;
#pragma unroll
    for (int o = 1; o < KG; o++) {
      f32x4 const *const other = reinterpret_cast<f32x4 const *>(smem + o * (STAGES * STAGE_ELEMS)) + wave * (TM * TN * 4 * 64) + lane;
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
          for (int g = 0; g < 4; g++) {
            f32x4 const v = other[((i * TN + j) * 4 + g) * 64];
#pragma unroll
            for (int e = 0; e < 4; e++) acc[i][j][4 * g + e] += v[e];
          }
    }
  }

  // Each wave stages its own WM x WN tile and writes it out in 16-byte chunks.
  bf16 *cs = smem + wave * (WM * CS);
  constexpr int CCH = WM * WN / 8 / 64;  // 16-byte chunks per lane
  // The activation is a compile-time functor here: a per-element switch inside
  // the unrolled loops made the epilogue several times longer than the GEMM's
  // own store traffic.
  auto finish = [&](auto actf) __attribute__((always_inline)) {
    bf16 *const dst = C;
    bool const add_old = accumulate != 0;
    // A wave stages and writes out its own tile, so only its own LDS accesses have to be ordered,
    // and those complete in program order: no barrier.  With one wave per SIMD (128x128 wave tiles)
    // the tile goes out in two halves of 64 rows, so that the stores of the first half are under
    // way while the second is converted.
    constexpr int HALVES = WIDE2 ? 2 : 1;
    constexpr int TMH = TM / HALVES;
#pragma unroll
    for (int half = 0; half < HALVES; half++) {
    // The lane's bias values depend on (j, g, lane / 32) only: they are
    // fetched once per (j, g) and used for the row blocks.
#pragma unroll
    for (int j = 0; j < TN; j++) {
#pragma unroll
      for (int g = 0; g < GROUPS; g++) {
        int const n = col_of(j, g);
        float bv[4];
        bias4(n0 + wn0 + n, bv);
#pragma unroll
        for (int i = half * TMH; i < (half + 1) * TMH; i++) {
          int const m = row_of(i);
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; e++) v[e] = acc[i][j][4 * g + e] + bv[e];
#pragma unroll
          for (int e = 0; e < 4; e++) v[e] = actf(v[e]);
          if (add_old) {
            // add the old value in fp32 before the single rounding
            bf16 const *const from = dst + (int64_t)(m0 + wm0 + m) * ldc + n0 + wn0 + n;
            u32x2 old = {0u, 0u};
            if constexpr (EDGE == kEdgeOverlap) {
              if (!TA || m0 + wm0 + m < M) old = load_any8(from);
            } else if constexpr (EDGE == kEdgeBounded) {
              int const left = m0 + wm0 + m < M ? N - (n0 + wn0 + n) : 0;  // columns of these four that exist
              old = left >= 4 ? load_any8(from) : left > 0 ? load_first4(from, left) : old;
            } else {
              old = *reinterpret_cast<u32x2 const *>(from);
            }
            v[0] += __uint_as_float(old[0] << 16);
            v[1] += __uint_as_float(old[0] & 0xffff0000u);
            v[2] += __uint_as_float(old[1] << 16);
            v[3] += __uint_as_float(old[1] & 0xffff0000u);
          }
          u32x2 w = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
          *reinterpret_cast<u32x2 *>(cs + m * CS + n) = w;
        }
      }
    }
#pragma unroll
    for (int i = half * (CCH / HALVES); i < (half + 1) * (CCH / HALVES); i++) {
      int c = lane + i * 64;
      int row = c / (WN / 8), ch = c % (WN / 8);
      u32x4 v = *reinterpret_cast<u32x4 const *>(cs + row * CS + ch * 8);
      put_piece(m0 + wm0 + row, n0 + wn0 + ch * 8, v, cs + row * CS + ch * 8);
    }
    }  // half
    if constexpr (kColsums) {
      if (tail.colsum_partials != nullptr) {  // uniform over the launch
        __syncthreads();
        column_sums(cs, CS, WM, WN, m0 + wm0, n0 + wn0, lane, 64);
      }
    }
  };
  if (!WIDE2 && partial != nullptr) {
    // raw accumulators, 16 bytes (4 consecutive columns) per store
    float *dst = partial + (int64_t)split * M * N;
#pragma unroll
    for (int i = 0; i < TM; i++) {
      int64_t const m = m0 + wm0 + row_of(i);
#pragma unroll
      for (int j = 0; j < TN; j++) {
#pragma unroll
        for (int g = 0; g < GROUPS; g++) {
          int const n = n0 + wn0 + col_of(j, g);
          if (EDGE != kEdgeNone && m >= M) continue;
          if (EDGE == kEdgeBounded && n >= N) continue;  // (N % 4 == 0 where a reduction is split)
          f32x4 v = {acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
          *reinterpret_cast<f32x4 *>(dst + m * N + n) = v;
        }
      }
    }
    return;
  }
  // One wave per SIMD with a 128x128 wave tile keeps 256 accumulator registers: neither an activation
  // nor a split reduction is compiled for it, so that nothing outside the loop competes for registers.
  if constexpr (WIDE2) {
    finish([](float v) { return v; });
    return;
  }
  if (act == FFK_ACT_NONE) {
    finish([](float v) { return v; });
  } else if (act == FFK_ACT_GELU) {
    finish([](float v) { return gelu_forward(v); });
  } else if (act == FFK_ACT_RELU) {
    finish([](float v) { return v >= 0.0f ? v : 0.0f; });
  } else {
    finish([act](float v) { return apply_activation(v, act); });
  }
}

// Second pass of split-K: C = epilogue(sum over splits of partial[s][M][N]).
static __global__ __launch_bounds__(256) void splitk_reduce_kernel(
    float const *__restrict__ partial, int splits, int M, int N, bf16 *C,
    int64_t ldc, bf16 const *__restrict__ bias, int act, int accumulate) {
  int64_t const q = (int64_t)blockIdx.x * 256 + threadIdx.x;
  int64_t const total = (int64_t)M * N;
  if (q * 4 >= total) return;
  int64_t const m = (q * 4) / N;
  int const n = (int)((q * 4) % N);
  f32x4 s = *reinterpret_cast<f32x4 const *>(partial + q * 4);
  for (int k = 1; k < splits; k++) {
    f32x4 v = *reinterpret_cast<f32x4 const *>(partial + k * total + q * 4);
    s += v;
  }
  bf16 *dst = C + m * ldc + n;
  float v[4] = {s[0], s[1], s[2], s[3]};
#pragma unroll
  for (int e = 0; e < 4; e++) {
    if (bias != nullptr) v[e] += VecIO<bf16>::load1(bias + n + e);
    v[e] = apply_activation(v[e], act);
  }
  if (accumulate) {
    u32x2 old = *reinterpret_cast<u32x2 const *>(dst);
    v[0] += __uint_as_float(old[0] << 16);
    v[1] += __uint_as_float(old[0] & 0xffff0000u);
    v[2] += __uint_as_float(old[1] << 16);
    v[3] += __uint_as_float(old[1] & 0xffff0000u);
  }
  u32x2 w = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
  *reinterpret_cast<u32x2 *>(dst) = w;
}

template <int BM, int BN, int WM, int WN, int BK, int STAGES>
struct PipeCfg {
  static constexpr int NW = (BM / WM) * (BN / WN);
  // (one wave per SIMD: five panels)
  static constexpr size_t kStageBytes = (size_t)(WM == 128 && STAGES == 2 ? 5 * (BM > BN ? BM : BN) : STAGES * (BM + BN)) * BK * sizeof(bf16);
  static constexpr size_t kOutBytes = (size_t)NW * WM * (WN + 8) * sizeof(bf16);
  static constexpr size_t kLds = kStageBytes > kOutBytes ? kStageBytes : kOutBytes;
  static_assert(kLds <= 160 * 1024, "LDS budget");
  // of KG groups of waves; groups of one wave keep the output tile behind their stages
  template <int KG>
  static constexpr size_t groups() {
    return KG == 1 ? kLds : KG * kStageBytes + (NW == 1 ? (size_t)BM * (BN + 8) * sizeof(bf16) : 0);
  }
};

template <int BM, int BN, int WM, int WN, int BK, int STAGES, int PF, bool TA, bool TB, int TAIL = 0, int EDGE = kEdgeNone,
          int KG = 1>
static hipError_t launch_pipe(hipStream_t st, bf16 const *A, bf16 const *B,
                              bf16 *C, int M, int N, int K, int64_t lda,
                              int64_t ldb, int64_t ldc, GemmEpilogue const &ep,
                              int splits = 1) {
  using Cfg = PipeCfg<BM, BN, WM, WN, BK, STAGES>;
  constexpr int NT = Cfg::NW * 64 * KG;
  constexpr size_t kLds = Cfg::template groups<KG>();
  static_assert(kLds <= 160 * 1024, "LDS budget");
  if (tl_name_sink != nullptr) {
    char rest[16] = "";  // EDGE and KG unless they have their default
    if (KG != 1) snprintf(rest, sizeof rest, ",%d,%d", EDGE, KG);
    else if (EDGE != kEdgeNone) snprintf(rest, sizeof rest, ",%d", EDGE);
    describe_only("gemm_bf16_pipe_kernel<%d,%d,%d,%d,%d,%d,%d,%s,%s,%d,false%s>", BM, BN, WM, WN, BK, STAGES, PF, tf(TA), tf(TB),
                  TAIL, rest);
    return hipSuccess;
  }
  auto kern = gemm_bf16_pipe_kernel<BM, BN, WM, WN, BK, STAGES, PF, TA, TB, TAIL, false, EDGE, KG>;
  GemmTailArgs const tail = {static_cast<bf16 const *>(ep.tail_in), static_cast<bf16 *>(ep.tail_out),
                             ep.tail_dropout, ep.tail_colsum_partials};
  static LdsOptIn lds;  // per template instance
  if (hipError_t e = lds.ensure(reinterpret_cast<void const *>(kern), (int)kLds); e != hipSuccess) return e;
  int const blocks = EDGE ? ((M + BM - 1) / BM) * ((N + BN - 1) / BN) : (M / BM) * (N / BN);
  if (splits > 1) {
    float *partial = static_cast<float *>(ep.splitk_ws);
    int const k_tiles = (K + BK - 1) / BK, per_split = (k_tiles + splits - 1) / splits;
    splits = (k_tiles + per_split - 1) / per_split;  // none is empty
    kern<<<blocks * splits, NT, kLds, st>>>(A, B, C, M, N, K, lda, ldb, ldc, nullptr, FFK_ACT_NONE, 0, partial, per_split,
                                            tail, GemmNoGroup{});
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    int64_t const quads = (int64_t)M * N / 4;
    splitk_reduce_kernel<<<(unsigned)ceil_div(quads, 256), 256, 0, st>>>(
        partial, splits, M, N, C, ldc, static_cast<bf16 const *>(ep.bias), ep.activation,
        ep.accumulate);
    return hipGetLastError();
  }
  kern<<<blocks, NT, kLds, st>>>(A, B, C, M, N, K, lda, ldb, ldc,
                                     static_cast<bf16 const *>(ep.bias), ep.activation,
                                     ep.accumulate, nullptr, 0, tail, GemmNoGroup{});
  return hipGetLastError();
}

// Several GEMMs of the same kind and reduction length in one launch.
template <int BM, int BN, int WM, int WN, int BK, int STAGES, int PF, bool TA, bool TB, int EDGE, int KG>
static hipError_t launch_pipe_group(hipStream_t st, GemmProblem const *p, int n, int K, bool accumulate, ColreduceBatch *sums) {
  using Cfg = PipeCfg<BM, BN, WM, WN, BK, STAGES>;
  constexpr int NT = Cfg::NW * 64 * KG;
  constexpr size_t kLds = Cfg::template groups<KG>();
  auto kern = gemm_bf16_pipe_kernel<BM, BN, WM, WN, BK, STAGES, PF, TA, TB, 0, true, EDGE, KG>;
  static LdsOptIn lds;
  if (hipError_t e = lds.ensure(reinterpret_cast<void const *>(kern), (int)kLds); e != hipSuccess) return e;
  GemmGroupArgs g = {};
  int64_t tiles = 0;
  for (int i = 0; i < n; i++) {
    if (i > 0) {
      g.p[i - 1] = {static_cast<bf16 const *>(p[i].A), static_cast<bf16 const *>(p[i].B), static_cast<bf16 *>(p[i].C),
                    p[i].lda, p[i].ldb, p[i].ldc, (int)p[i].M, (int)p[i].N, (int)tiles};
    }
    tiles += ceil_div(p[i].M, BM) * ceil_div(p[i].N, BN);
  }
  g.count = n - 1;
  g.first_sum = (int)tiles;
  if (sums != nullptr && sums->count > 0 && sums->dtype == FFK_BF16) {
    g.sums = *sums;
    tiles += colreduce_blocks(*sums);
    sums->count = 0;
  }
  kern<<<(unsigned)tiles, NT, kLds, st>>>(static_cast<bf16 const *>(p[0].A), static_cast<bf16 const *>(p[0].B),
                                         static_cast<bf16 *>(p[0].C), (int)p[0].M, (int)p[0].N, K, p[0].lda, p[0].ldb,
                                         p[0].ldc, nullptr, FFK_ACT_NONE, accumulate ? 1 : 0, nullptr, 0, GemmTailArgs{}, g);
  return hipGetLastError();
}

template <int BM, int BN, int WM, int WN, bool TA, bool TB>
static hipError_t launch_bf16(hipStream_t st, bf16 const *A, bf16 const *B,
                              bf16 *C, int M, int N, int K, int64_t lda,
                              int64_t ldb, int64_t ldc, GemmEpilogue const &ep) {
  int const blocks = (int)(ceil_div(M, BM) * ceil_div(N, BN));
  constexpr int NT = (BM / WM) * (BN / WN) * 64;
  bf16 const *bias = static_cast<bf16 const *>(ep.bias);
  if (describe_only("gemm_bf16_kernel<%d,%d,%d,%d,%s,%s>", BM, BN, WM, WN, tf(TA), tf(TB))) return hipSuccess;
  gemm_bf16_kernel<BM, BN, WM, WN, TA, TB><<<blocks, NT, 0, st>>>(A, B, C, M, N, K, lda, ldb, ldc, bias, ep.activation,
                                                                ep.accumulate);
  return hipGetLastError();
}

// FFK_OPTION_GEMM_VARIANT forces a tile (EdgeTile's values, 192, or 1 = the
// register-staged kernel); 0 = the heuristic.  For tuning runs and tests.
inline int gemm_variant_override() { return option(FFK_OPTION_GEMM_VARIANT); }

// What every pipelined kernel asks of the operands, whatever its tile.
inline bool pipe_operands_ok(bf16 const *C, int K, int64_t lda, int64_t ldb, int64_t ldc, GemmEpilogue const &ep) {
  bool const c_vec = (ldc % 8 == 0) && aligned16(C);
  // the pipelined kernels fetch the bias in 8-byte pieces
  bool const aux_ok = reinterpret_cast<uintptr_t>(ep.bias) % 8 == 0;
  // the direct loads address an operand panel with 32-bit byte offsets
  bool const panel_ok = 2 * 256 * std::max(lda, ldb) < (int64_t(1) << 31);
  return c_vec && aux_ok && panel_ok && K % 64 == 0;
}

// Which pipelined tile a bf16 GEMM runs on: 256, 128, or 0 (none of the two:
// split-K or the register-staged kernels).
inline int pipe_tile_for(bf16 const *C, int M, int N, int K, int64_t lda, int64_t ldb, int64_t ldc,
                         GemmEpilogue const &ep, int variant) {
  if (!pipe_operands_ok(C, K, lda, ldb, ldc, ep) || variant == 1) return 0;
  bool const fits256 = M % 256 == 0 && N % 256 == 0;
  bool const fits128 = M % 128 == 0 && N % 128 == 0;
  int64_t const t256 = fits256 ? (int64_t)(M / 256) * (N / 256) : 0;
  int64_t const t128 = fits128 ? (int64_t)(M / 128) * (N / 128) : 0;
  // 256x256 tiles (8 waves of 128x64, four 32-deep stages of 32 KB whose
  // refills are spread over the k-steps) halve the L2->LDS traffic per flop;
  // they win whenever they still occupy most CUs.  Otherwise 128x128x64 tiles
  // with 8 waves of 64x32 keep two waves per SIMD on every CU.
  if ((variant == 0 && t256 >= kNumCU * 3 / 4) || ((variant == 256 || variant == 264) && fits256)) return 256;
  if ((variant == 0 && t128 >= kNumCU / 2) || (variant == 128 && fits128)) return 128;
  return 0;
}

// What the pipelined kernels ask of operands that do not divide into tiles: panels that 32-bit byte
// offsets reach.
inline bool edge_operands_ok(int64_t lda, int64_t ldb) { return 2 * 256 * std::max(lda, ldb) < (int64_t(1) << 31); }

// The time of a bf16 product on each of the tiles, in us, from which its tile is chosen.  Its
// coefficients are those with which the tiles picked for 670 products drawn from M 64-5000, N and K 128-4096
// took least: 1.4% longer than the best tile each on these and on 330 others (2.4% before, 20% and more at
// the worst, of 2048-long reductions and of 257 to 512 tiles of 64 x 64: 1149 x 768 over 2048 12.7 -> 10.5 us, 828 x
// 1536 over 2560 21.5 -> 18.1).  It ranks the tiles and does not predict: launch to launch they took 0.8 to 2.1 times
// its figure (median 1.3; 2-3 us of each is the launch), the short and the transposed ones most.
// The fit is of the 256-wide tiles on 32x32x16 matrix instructions; on 16x16x32 they take some 8% less.  Of 240 other
// products drawn from M 64-5000, N and K 128-4096 on the present kernels, the tile picked takes 2.4% longer than the best
// one, and of the 52 with 4 M outputs and reductions of 1024 and more 5.3%: never where the wide tile is the best (13
// products), most where 256 x 128 tiles would be and gemm_takes_256x128 does not hold (1432 x 3152 over 3528 72 us, 52 on those).
//  - a round over the chip costs its 64-deep k-tiles times what one takes with so many CUs busy
//    (memory and LDS are shared, the clock too), and a constant of filling, draining and storing
//  - 32 x 32, four waves that split the reduction, two workgroups a CU
//    64 x 64, two groups of waves that split the reduction, two workgroups a CU
//    64 x 64 deep: four LDS stages a group, one workgroup a CU: holds its rate where the operands
//    come from behind L2, as they do in reductions of 2048 and longer
//    128 x 64: eight waves, two workgroups a CU; 128 x 128; 256 x 256; wide: the latter with one wave
//    per SIMD
enum EdgeTile { kTile32 = 32, kTile64 = 64, kTile64Deep = 65, kTile128x64 = 70, kTile128 = 128, kTile256x128 = 130, kTile256 = 256, kTile256Wide = 264 };
inline double gemm_tile_us(EdgeTile t, double m, double n, double k, double splits = 1) {
  int const bm = t == kTile32 ? 32 : t == kTile64 || t == kTile64Deep ? 64 : t == kTile128x64 || t == kTile128 ? 128 : 256;
  int const bn = t == kTile128x64 ? 64 : t == kTile256x128 ? 128 : bm;
  double const tiles = ceil(m / bm) * ceil(n / bn) * splits, kt = ceil(ceil(k / 64) / splits);
  auto round_us = [&](double count) {  // of `count` workgroups at a time
    double const f = count / kNumCU;
    switch (t) {
      case kTile32: return f <= 1 ? kt * 0.11 + 1.9 : kt * 0.40 + 2.4;
      case kTile64: return f <= 1 ? kt * 0.166 + 1.8 : kt * 0.28 + 1.9;
      case kTile64Deep: return kt * 0.167 + 2.1;
      case kTile128x64: return f <= 1 ? kt * (0.30 + 0.06 * f) + 1.55 : kt * 0.63 + 2.35;
      case kTile128: return kt * std::max(0.325, 0.11 + 0.367 * f) + 2.1;
      case kTile256x128: return kt * (0.42 + 0.40 * f) + 3.5;
      case kTile256: return kt * std::max(1.09, 0.35 + 1.25 * f) + 5.5 + 2.0 * f;
      default: return kt * std::max(0.96, 0.25 + 1.19 * f) + 5.5 + 3.0 * f;
    }
  };
  double const a_round = t == kTile32 || t == kTile64 || t == kTile128x64 ? 2 * kNumCU : kNumCU;
  double const full = floor(tiles / a_round), last = tiles - full * a_round;
  double us = full * round_us(a_round) + (last > 0 ? round_us(last) : 0.0);
  // the rounds of 128 x 128 tiles overlap less than the first one's fill suggests
  if (t == kTile128) us += 1.9 * (ceil(tiles / a_round) - 1);
  if (t == kTile64 && kt > 30) us += 0.2 * (kt - 30) * ceil(tiles / a_round);
  if (splits > 1) us += 4.0 + splits * m * n * 8 / 4.0e6;  // the partial sums: written and read at 4 TB/s
  return us;
}
// 256 x 128 tiles, eight waves of 64 x 64, where one round holds them and two of 128 x 128 were needed: both tiles
// have one workgroup a CU, and this one does with 48 KB of loads and 128 of LDS reads a 64-deep k-tile what two of the
// other do with 64 and 192.  Launch to launch, 1379 x 3072 over 768 16.9 -> 14.6 us, 3571 x 2048 over 512 15.2 -> 12.5,
// 2176 x 2048 over 2048 33 -> 29.  The fuller the round and the longer the reduction, the more the CUs share one limit, of
// memory and clock: 3200 x 2048 over 1024 19.8 and 20.5, 2816 x 2048 over 2048 with A transposed 33.8 and 35.1, which is
// where the line lies; 4096 x 1024 over 4096, 128 of these tiles, 51 where 256 of the others take 32.
inline bool gemm_takes_256x128(int M, int N, int K) {
  int64_t const t128 = ceil_div(M, 128) * ceil_div(N, 128), tiles = ceil_div(M, 256) * ceil_div(N, 128);
  return M >= 256 && N >= 128 && t128 > kNumCU && tiles <= kNumCU && K <= 2048 && (2 * tiles - kNumCU) * K <= 512 * kNumCU;
}
inline EdgeTile gemm_tile_for(int M, int N, int K, bool wide_ok, double *time = nullptr) {
  if (gemm_takes_256x128(M, N, K)) {
    if (time != nullptr) *time = gemm_tile_us(kTile256x128, M, N, K);
    return kTile256x128;
  }
  EdgeTile best = kTile64;
  double least = gemm_tile_us(kTile64, M, N, K);
  for (EdgeTile const t : {kTile32, kTile64Deep, kTile128x64, kTile128, kTile256, kTile256Wide}) {
    if ((t == kTile256Wide) != (wide_ok && K >= 1024) && (t == kTile256Wide || t == kTile256)) continue;
    double const us = gemm_tile_us(t, M, N, K);
    if (us < least) best = t, least = us;
  }
  if (time != nullptr) *time = least;
  return best;
}

// The tile of the plain kernel for this problem if it is one of those whose waves split the reduction (an
// epilogue's tail then has to run on that tile too for the same bits), 0 if it is one of the larger ones,
// which all add up in the same order.
inline int gemm_split_tile(int M, int N, int K, GemmEpilogue const &ep) {
  EdgeTile const t = gemm_tile_for(M, N, K, ep.activation == FFK_ACT_NONE);
  if (t == kTile32 || t == kTile64 || t == kTile64Deep) return t;
  if (t == kTile256x128) return 0;
  int const bm = t == kTile256 || t == kTile256Wide ? 256 : 128, bn = t == kTile128x64 ? 64 : bm;
  return M < bm || N < bn ? kTile64 : 0;
}

// Splitting the reduction over workgroups, where there is scratch for it: 128 x 128 or 256 x 256 tiles
// in as many splits as make the product fastest.  1: none does.  (Reductions worth splitting stream
// their operands from memory, which 256 x 256 tiles read half as often: [2048, 50257] . [50257, 1024]
// takes 446 us unsplit, 290 us on 128 x 128 tiles and 2 splits, 210 us on 256 x 256 tiles and 8.)
inline int gemm_splits_for(int M, int N, int K, size_t scratch, double unsplit_us, EdgeTile &tile) {
  int best = 1;
  double least = unsplit_us;
  for (EdgeTile const t : {kTile128, kTile256}) {
    if (M < t || N < t) continue;
    for (int s = 2; s <= 16 && ceil_div(K, 64) >= 8 * s && (size_t)s * M * N * sizeof(float) <= scratch; s *= 2) {
      double const us = gemm_tile_us(t, M, N, K, s) * (t == kTile128 ? 1.2 : 1.0);
      if (us < least) best = s, least = us, tile = t;
    }
  }
  return best;
}

// A product whose last round of 256 x 256 tiles is nearly empty: the rows (along_m) or columns that make
// whole rounds go first, the others as a product of their own on the tile that suits them.  How many
// rows or columns the first one takes, 0 if one launch is as soon done.  ([2048, 1024] . [50257, 1024]^T
// is 1576 tiles, six rounds and 40 more: 238 us, 214 in two launches.)
inline int gemm_whole_rounds(int M, int N, int K, bool wide_ok, double one_launch_us, bool &along_m) {
  EdgeTile const t = wide_ok && K >= 1024 ? kTile256Wide : kTile256;
  int64_t const nbm = ceil_div(M, 256), nbn = ceil_div(N, 256), full = nbm * nbn / kNumCU * kNumCU;
  if (full == 0 || full == nbm * nbn) return 0;
  int first = 0;
  double least = one_launch_us - 2.0;
  for (bool const m : {false, true}) {
    int64_t const lines = full / (m ? nbn : nbm) * 256;
    if (lines == 0 || lines >= (m ? M : N)) continue;
    double rest = 0;
    gemm_tile_for(m ? M - (int)lines : M, m ? N : N - (int)lines, K, wide_ok, &rest);
    double const us = gemm_tile_us(t, m ? (double)lines : M, m ? N : (double)lines, K) + rest + 3.0;
    if (us < least) first = (int)lines, along_m = m, least = us;
  }
  return first;
}

// A GEMM with element-wise operators on its tile store.  gemm_tail_supported has been asked.
template <int TAIL, bool TA, bool TB>
static hipError_t launch_tail(hipStream_t st, bf16 const *A, bf16 const *B, bf16 *C, int M, int N, int K, int64_t lda,
                              int64_t ldb, int64_t ldc, GemmEpilogue const &ep) {
  // column sums are taken over blocks of 32 rows from multiples of 32 on, where overlapping tiles do not begin
  constexpr bool sums = TAIL == GemmEpilogue::kTailDropoutGeluGrad || TAIL == GemmEpilogue::kTailDropoutReluGrad;
  constexpr int edge = sums ? kEdgeBounded : kEdgeOverlap;
  int const variant = gemm_variant_override();
  if (variant == 0 && gemm_takes_256x128(M, N, K)) {
    if (M % 256 == 0 && N % 128 == 0 && pipe_operands_ok(C, K, lda, ldb, ldc, ep)) {
      return launch_pipe<256, 128, 64, 64, 64, 3, 1, TA, TB, TAIL>(st, A, B, C, M, N, K, lda, ldb, ldc, ep);
    }
    return launch_pipe<256, 128, 64, 64, 64, 3, 1, TA, TB, TAIL, edge>(st, A, B, C, M, N, K, lda, ldb, ldc, ep);
  }
  int const tile = pipe_tile_for(C, M, N, K, lda, ldb, ldc, ep, variant);
  if (tile == 256) return launch_pipe<256, 256, 128, 64, 32, 4, 1, TA, TB, TAIL>(st, A, B, C, M, N, K, lda, ldb, ldc, ep);
  if (tile == 128) return launch_pipe<128, 128, 64, 32, 64, 4, 1, TA, TB, TAIL>(st, A, B, C, M, N, K, lda, ldb, ldc, ep);
  switch (gemm_split_tile(M, N, K, ep)) {
    case kTile32: return launch_pipe<32, 32, 32, 32, 32, 4, 1, TA, TB, TAIL, kEdgeBounded, 4>(st, A, B, C, M, N, K, lda, ldb, ldc, ep);
    case kTile64: return launch_pipe<64, 64, 32, 32, 64, 2, 3, TA, TB, TAIL, kEdgeBounded, 2>(st, A, B, C, M, N, K, lda, ldb, ldc, ep);
    case kTile64Deep: return launch_pipe<64, 64, 32, 32, 64, 4, 3, TA, TB, TAIL, kEdgeBounded, 2>(st, A, B, C, M, N, K, lda, ldb, ldc, ep);
  }
  if constexpr (TAIL == GemmEpilogue::kTailGeluDropout) {
    return hipErrorInvalidValue;  // (one large tile a CU: gemm_tail_supported has refused it)
  } else {
    if (!sums && (M < 128 || N < 128)) return hipErrorInvalidValue;
    // 128 x 64 where the plain product takes it (1379 x 3072 over 768 with ReLU and dropout: 24.4 -> 21.6 us), and
    // where a round holds them all: the operators on the store are then spread over twice the CUs (1379 x 768
    // over 3072 with dropout and add: 25.7 -> 22.7).
    if constexpr (!sums) {
      if (gemm_tile_for(M, N, K, ep.activation == FFK_ACT_NONE) == kTile128x64 ||
          ceil_div(M, 128) * ceil_div(N, 64) <= kNumCU) {
        return launch_pipe<128, 64, 32, 32, 64, 3, 1, TA, TB, TAIL, edge>(st, A, B, C, M, N, K, lda, ldb, ldc, ep);
      }
    }
    return launch_pipe<128, 128, 64, 32, 64, 4, 1, TA, TB, TAIL, edge>(st, A, B, C, M, N, K, lda, ldb, ldc, ep);
  }
}
template <bool TA, bool TB>
hipError_t pick_bf16_tail(hipStream_t st, bf16 const *A, bf16 const *B, bf16 *C, int M, int N, int K, int64_t lda,
                          int64_t ldb, int64_t ldc, GemmEpilogue const &ep) {
  switch (ep.tail) {
    case GemmEpilogue::kTailDropoutAdd:
      return launch_tail<GemmEpilogue::kTailDropoutAdd, TA, TB>(st, A, B, C, M, N, K, lda, ldb, ldc, ep);
    case GemmEpilogue::kTailGeluDropout:
      if constexpr (TB) return launch_tail<GemmEpilogue::kTailGeluDropout, TA, TB>(st, A, B, C, M, N, K, lda, ldb, ldc, ep);
      break;
    case GemmEpilogue::kTailActDropout:
      if constexpr (TB) return launch_tail<GemmEpilogue::kTailActDropout, TA, TB>(st, A, B, C, M, N, K, lda, ldb, ldc, ep);
      break;
    case GemmEpilogue::kTailDropoutGeluGrad:
      if constexpr (!TB) return launch_tail<GemmEpilogue::kTailDropoutGeluGrad, TA, TB>(st, A, B, C, M, N, K, lda, ldb, ldc, ep);
      break;
    case GemmEpilogue::kTailDropoutReluGrad:
      if constexpr (!TB) return launch_tail<GemmEpilogue::kTailDropoutReluGrad, TA, TB>(st, A, B, C, M, N, K, lda, ldb, ldc, ep);
      break;
  }
  return hipErrorInvalidValue;
}

// A group of problems that each leave part of the chip idle: 128x128 tiles, 64x64 or 32x32 ones, whichever
// takes less for all of them together by formulas of the group's own, rounds times k-tiles.  They
// rank the three and do not predict: 432 tiles of 128 x 128 over 1379 rows (the gradients of a 768-wide
// layer) 37 us, 22 by the formula.
template <bool TA, bool TB>
hipError_t pick_bf16_group(hipStream_t st, GemmProblem const *p, int n, int K, bool accumulate, ColreduceBatch *sums) {
  bool exact = K % 64 == 0, fits = true, exact256 = true;
  double t32 = 0, t64 = 0, t128 = 0;
  for (int i = 0; i < n; i++) {
    exact = exact && p[i].M % 128 == 0 && p[i].N % 128 == 0 && p[i].ldc % 8 == 0 && aligned16(p[i].C);
    exact256 = exact256 && p[i].M % 256 == 0 && p[i].N % 256 == 0;
    fits = fits && p[i].M >= 128 && p[i].N >= 128 && !(accumulate && p[i].N % 8 != 0);
    t32 += (double)(ceil_div(p[i].M, 32) * ceil_div(p[i].N, 32));
    t64 += (double)(ceil_div(p[i].M, 64) * ceil_div(p[i].N, 64));
    t128 += (double)(ceil_div(p[i].M, 128) * ceil_div(p[i].N, 128));
  }
  double const kt = (double)ceil_div(K, 64);
  bool const deep = t64 <= kNumCU && kt > 32;
  double const us64 = deep ? kt * 0.23 + 2.0 : t64 <= kNumCU ? kt * 0.17 + 1.0
                    : kt > 32 ? kt * 0.285 * t64 / kNumCU + 1.0 : ceil(t64 / (2 * kNumCU)) * (kt * 0.39 + 1.0);
  double const us128 = ceil(t128 / kNumCU) * (kt * 0.46 + 1.0);
  double const us32 = t32 <= kNumCU ? kt * (kt > 32 ? 0.18 : 0.11) + 1.0 : t32 <= 2 * kNumCU ? kt * (kt > 32 ? 0.36 : 0.22) + 1.0 : 1e9;
  if (us32 < us64 && (us32 < us128 || !fits)) return launch_pipe_group<32, 32, 32, 32, 32, 4, 1, TA, TB, kEdgeBounded, 4>(st, p, n, K, accumulate, sums);
  if (!fits || us64 < us128) {
    // (long reductions on four LDS stages a group of waves, one workgroup a CU: 512 x 2048 over 8065, 256 tiles, 49
    // us on two)
    if (deep) return launch_pipe_group<64, 64, 32, 32, 64, 4, 3, TA, TB, kEdgeBounded, 2>(st, p, n, K, accumulate, sums);
    return launch_pipe_group<64, 64, 32, 32, 64, 2, 3, TA, TB, kEdgeBounded, 2>(st, p, n, K, accumulate, sums);
  }
  // Long reductions of whole 256 x 256 tiles: a round of them, three quarters full, takes less than three
  // of 128 x 128 (four gradients of 12.6 M elements together over 4096
  // rows: 106-114 us against 119; 81 by the model).
  if (exact && exact256 && K >= 1024 &&
      gemm_tile_us(kTile256Wide, 64 * t128, 256, K) < gemm_tile_us(kTile128, 128 * t128, 128, K)) {
    return launch_pipe_group<256, 256, 128, 128, 64, 2, 1, TA, TB, kEdgeNone, 1>(st, p, n, K, accumulate, sums);
  }
  if (exact) return launch_pipe_group<128, 128, 64, 32, 64, 4, 1, TA, TB, kEdgeNone, 1>(st, p, n, K, accumulate, sums);
  return launch_pipe_group<128, 128, 64, 32, 64, 4, 1, TA, TB, kEdgeOverlap, 1>(st, p, n, K, accumulate, sums);
}

template <bool TA, bool TB>
hipError_t pick_bf16(hipStream_t st, bf16 const *A, bf16 const *B,
                            bf16 *C, int M, int N, int K, int64_t lda,
                            int64_t ldb, int64_t ldc, GemmEpilogue const &ep, bool vec) {
  int const variant = vec ? gemm_variant_override() : 1;  // 1: the register-staged kernel, whose loads take any address
  // An output that 256x256 tiles cover in a ragged last round but 256x192 tiles cover in whole
  // rounds of the chip (the attention block's fused Q/K/V projection: [4096, 3072] is 192 tiles of
  // the first kind on 256 CUs, 256 of the second): one wave per SIMD on 128x96 wave tiles.  Only
  // with both operands K-contiguous: a [K][192] panel does not divide into whole direct loads.
  if constexpr (!TA && TB) {
    bool const fits192 = M % 256 == 0 && N % 192 == 0;
    int64_t const t256 = M % 256 == 0 && N % 256 == 0 ? (int64_t)(M / 256) * (N / 256) : 0;
    int64_t const t192 = fits192 ? (int64_t)(M / 256) * (N / 192) : 0;
    bool const whole_rounds = t192 > 0 && t192 % kNumCU == 0 && t256 % kNumCU != 0;
    if (pipe_operands_ok(C, K, lda, ldb, ldc, ep) && variant != 1 && ep.activation == FFK_ACT_NONE && K >= 1024 &&
        (variant == 192 ? fits192 : (variant == 0 && whole_rounds))) {
      return launch_pipe<256, 192, 128, 96, 64, 2, 1, TA, TB>(st, A, B, C, M, N, K, lda, ldb, ldc, ep);
    }
  }
  if (variant != 1 && edge_operands_ok(lda, ldb)) {
    bool const wide_ok = ep.activation == FFK_ACT_NONE && ldc % 8 == 0;
    double us;
    EdgeTile tile = gemm_tile_for(M, N, K, wide_ok, &us);
    bool const forced = variant == 32 || variant == 64 || variant == 65 || variant == 70 || variant == 128 || variant == 130 || variant == 256 || variant == 264;
    bool const whole128 = M % 128 == 0 && N % 128 == 0 && pipe_operands_ok(C, K, lda, ldb, ldc, ep);
    if (forced) {
      tile = variant == kTile256Wide && ep.activation != FFK_ACT_NONE ? kTile256 : (EdgeTile)variant;
    } else {
      if (ep.splitk_ws != nullptr && aligned16(ep.splitk_ws) && aligned16(C) && N % 8 == 0 && ldc % 8 == 0) {
        EdgeTile split_tile = tile;
        int const splits = gemm_splits_for(M, N, K, ep.splitk_ws_bytes, us, split_tile);
        if (splits > 1) {
          if (split_tile == kTile256) {
            return launch_pipe<256, 256, 128, 64, 32, 4, 1, TA, TB, 0, kEdgeOverlap>(st, A, B, C, M, N, K, lda, ldb, ldc, ep, splits);
          }
          if (whole128) return launch_pipe<128, 128, 64, 32, 64, 4, 1, TA, TB>(st, A, B, C, M, N, K, lda, ldb, ldc, ep, splits);
          return launch_pipe<128, 128, 64, 32, 64, 4, 1, TA, TB, 0, kEdgeOverlap>(st, A, B, C, M, N, K, lda, ldb, ldc, ep, splits);
        }
      }
      // A long reduction over whole tiles stays on this tile, which tests name: 1024 x 2048 over 4096 25-28 us, 27-35
      // on 64-wide ones; but 1024 x 1024, where the deep 64-wide tile would be faster, 24-27 us, 17-19 on that.  Not
      // where that one saves more than as much: 2048 x 512 over 8064 50 us, 31.  And one that gives half the CUs
      // such a tile, on which operators on its store would run, adds up in their order.
      int64_t const t128 = (int64_t)(M / 128) * (N / 128);
      if (whole128 && (tile == kTile64 || tile == kTile64Deep) &&
          (t128 >= kNumCU / 2 || (t128 >= kNumCU / 4 && K >= 4096 && gemm_tile_us(kTile128, M, N, K) - us < 12.0))) {
        tile = kTile128;
      }
      bool along_m = false;
      int const first = M >= 256 && N >= 256 ? gemm_whole_rounds(M, N, K, wide_ok, us, along_m) : 0;
      if (first > 0) {
        GemmEpilogue rest = ep;
        int const m = along_m ? first : 0, n = along_m ? 0 : first;
        if (ep.bias != nullptr) rest.bias = static_cast<bf16 const *>(ep.bias) + n;
        hipError_t const e = pick_bf16<TA, TB>(st, A + (TA ? (int64_t)m : m * lda), B + (TB ? n * ldb : (int64_t)n), C + m * ldc + n,
                                               M - m, N - n, K, lda, ldb, ldc, rest, vec);
        if (e != hipSuccess) return e;
        return pick_bf16<TA, TB>(st, A, B, C, along_m ? first : M, along_m ? N : first, K, lda, ldb, ldc, ep, vec);
      }
    }
    // tiles that begin early: the output has to hold one, and old values added by one workgroup only
    int const bm = tile == kTile256 || tile == kTile256x128 || tile == kTile256Wide ? 256 : 128;
    int const bn = tile == kTile128x64 ? 64 : tile == kTile256x128 ? 128 : bm;
    if (tile != kTile32 && tile != kTile64 && tile != kTile64Deep && (M < bm || N < bn || (ep.accumulate && N % 8 != 0))) tile = kTile64;
    bool const whole = M % bm == 0 && N % bn == 0 && pipe_operands_ok(C, K, lda, ldb, ldc, ep);
    switch (tile) {
      case kTile256Wide:
        if (whole) return launch_pipe<256, 256, 128, 128, 64, 2, 1, TA, TB>(st, A, B, C, M, N, K, lda, ldb, ldc, ep);
        return launch_pipe<256, 256, 128, 128, 64, 2, 1, TA, TB, 0, kEdgeOverlap>(st, A, B, C, M, N, K, lda, ldb, ldc, ep);
      case kTile256:
        if (whole) return launch_pipe<256, 256, 128, 64, 32, 4, 1, TA, TB>(st, A, B, C, M, N, K, lda, ldb, ldc, ep);
        return launch_pipe<256, 256, 128, 64, 32, 4, 1, TA, TB, 0, kEdgeOverlap>(st, A, B, C, M, N, K, lda, ldb, ldc, ep);
      case kTile256x128:
        if (whole) return launch_pipe<256, 128, 64, 64, 64, 3, 1, TA, TB>(st, A, B, C, M, N, K, lda, ldb, ldc, ep);
        return launch_pipe<256, 128, 64, 64, 64, 3, 1, TA, TB, 0, kEdgeOverlap>(st, A, B, C, M, N, K, lda, ldb, ldc, ep);
      case kTile128:
        if (whole) return launch_pipe<128, 128, 64, 32, 64, 4, 1, TA, TB>(st, A, B, C, M, N, K, lda, ldb, ldc, ep);
        return launch_pipe<128, 128, 64, 32, 64, 4, 1, TA, TB, 0, kEdgeOverlap>(st, A, B, C, M, N, K, lda, ldb, ldc, ep);
      case kTile128x64:
        return launch_pipe<128, 64, 32, 32, 64, 3, 1, TA, TB, 0, kEdgeOverlap>(st, A, B, C, M, N, K, lda, ldb, ldc, ep);
      case kTile64Deep:
        return launch_pipe<64, 64, 32, 32, 64, 4, 3, TA, TB, 0, kEdgeBounded, 2>(st, A, B, C, M, N, K, lda, ldb, ldc, ep);
      case kTile32:
        return launch_pipe<32, 32, 32, 32, 32, 4, 1, TA, TB, 0, kEdgeBounded, 4>(st, A, B, C, M, N, K, lda, ldb, ldc, ep);
      case kTile64:
        return launch_pipe<64, 64, 32, 32, 64, 2, 3, TA, TB, 0, kEdgeBounded, 2>(st, A, B, C, M, N, K, lda, ldb, ldc, ep);
    }
  }
  // By what a k-tile takes of a CU: on a 64x64 tile 0.42 us among others and 0.62 alone, on a 128x128 one 0.85
  // and 1.0 ([2560, 2479] . [1324, 2479]^T 60 us on the first, 51 on the second; [1024, 1023] . [1023, 1023] 16 on
  // the first, with a quarter of the chip in use on the second).
  double const per_cu64 = (double)(ceil_div(M, 64) * ceil_div(N, 64)) / kNumCU;
  double const rounds128 = ceil((double)(ceil_div(M, 128) * ceil_div(N, 128)) / kNumCU);
  if (std::max(1.0, 0.85 * rounds128) < std::max(0.62, 0.42 * per_cu64)) {
    return launch_bf16<128, 128, 64, 32, TA, TB>(st, A, B, C, M, N, K, lda, ldb, ldc, ep);
  }
  return launch_bf16<64, 64, 32, 32, TA, TB>(st, A, B, C, M, N, K, lda, ldb, ldc, ep);
}


}  // namespace ffk
