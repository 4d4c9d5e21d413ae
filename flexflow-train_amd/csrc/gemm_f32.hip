// fp32 GEMM kernels for gfx950 (v_mfma_f32_32x32x2f32), behind gemm_dispatch.
#include <algorithm>
#include "gemm_bf16.h"
#include "small_f32.h"

namespace ffk {

// ---------------------------------------------------------------------------
// fp32 MFMA kernel (32x32x2), 64x64 block tile, bounds-checked everywhere.
// ---------------------------------------------------------------------------
template <bool TA, bool TB>
__global__ __launch_bounds__(256) void gemm_f32_kernel(
    float const *__restrict__ A, float const *__restrict__ B, float *C, int M,
    int N, int K, int64_t lda, int64_t ldb, int64_t ldc,
    float const *__restrict__ bias, int act, int accumulate) {
  constexpr int BM = 64, BN = 64, BKF = 16, LD = 68;
  __shared__ float As[BKF][LD];  // [k][m]
  __shared__ float Bs[BKF][LD];  // [k][n]
  int const t = threadIdx.x;
  int const lane = t & 63;
  int const wave = t >> 6;
  int const wm0 = (wave >> 1) * 32;
  int const wn0 = (wave & 1) * 32;
  int const nbn = (N + BN - 1) / BN;
  int const m0 = (blockIdx.x / nbn) * BM;
  int const n0 = (blockIdx.x % nbn) * BN;

  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; r++) acc[r] = 0.0f;

  for (int k0 = 0; k0 < K; k0 += BKF) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      int m, k;
      if (!TA) {  // A[M,K]: k fastest across lanes
        k = t & 15;
        m = (t >> 4) + 16 * i;
      } else {  // A[K,M]: m fastest
        m = t & 63;
        k = (t >> 6) + 4 * i;
      }
      int gm = m0 + m, gk = k0 + k;
      float v = 0.0f;
      if (gm < M && gk < K) {
        v = TA ? A[(int64_t)gk * lda + gm] : A[(int64_t)gm * lda + gk];
      }
      As[k][m] = v;
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
      int n, k;
      if (TB) {  // B[N,K]: k fastest
        k = t & 15;
        n = (t >> 4) + 16 * i;
      } else {  // B[K,N]: n fastest
        n = t & 63;
        k = (t >> 6) + 4 * i;
      }
      int gn = n0 + n, gk = k0 + k;
      float v = 0.0f;
      if (gn < N && gk < K) {
        v = TB ? B[(int64_t)gn * ldb + gk] : B[(int64_t)gk * ldb + gn];
      }
      Bs[k][n] = v;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < BKF / 2; kk++) {
      float a = As[2 * kk + (lane >> 5)][wm0 + (lane & 31)];
      float b = Bs[2 * kk + (lane >> 5)][wn0 + (lane & 31)];
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc, 0, 0, 0);
    }
    __syncthreads();
  }

  int const n = n0 + wn0 + (lane & 31);
  if (n < N) {
    float bv = bias != nullptr ? bias[n] : 0.0f;
#pragma unroll
    for (int r = 0; r < 16; r++) {
      int const m = m0 + wm0 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
      if (m < M) {
        float v = apply_activation(acc[r] + bv, act);
        float *dst = C + (int64_t)m * ldc + n;
        if (accumulate) {
          v += *dst;
        }
        *dst = v;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// fp32 MFMA kernel: BM x BN block tile (128 or 64 each), 2 x 2 waves of BM/2 x BN/2, reduction
// tiles of 32, operands read 16 bytes at a time.
// The next tile travels global -> registers while this one is multiplied and
// goes to the other LDS buffer afterwards: one barrier per tile.  The fp32
// MFMA (32x32x2, 64 cycles) is so slow next to its two one-register operands
// that LDS and issue bandwidth are never short; what the kernel has to do is
// keep loads in flight and the matrix pipe fed, which two workgroups per CU and
// fragments read one step ahead take care of.
//   An operand whose reduction index is contiguous in memory (A[M,K], B[N,K])
// lies in LDS as [k / 2][row][k % 2], row stride 2 * rows + 4: a lane's four
// consecutive k go out as two 8-byte writes, and the MFMA read -- lanes 0-31
// one k, lanes 32-63 the next -- touches 64 consecutive floats.  The compiler
// pairs a lane's reads for two 32-row blocks into one two-dword read, which is
// served 32 lanes at a time: the pairs of odd blocks are stored swapped, so
// that those 32 lanes take even banks for one block and odd banks for the
// other (unswapped they met in the same banks: 2.6 conflict cycles per cycle
// of LDS work, the matrix pipe 80% busy).  An operand
// whose rows are contiguous (A[K,M], B[K,N]) lies as [k][row] with the two
// 32-float halves of every odd k swapped, which does the same for the read
// without padding.  A group of waves (KG below) adds every element's products in
// ascending k, two per MFMA, as gemm_f32_kernel does: with one group the two
// kernels give the same bits.
// Rows and columns past the edge are read from the last valid ones and never
// stored; k past the end is zeroed when the tile is written to LDS.
// KG: groups of four waves that split the k-tiles, each with LDS buffers of its own, and add up at the end.
// ANY: lengths and row starts that are no multiple of four elements.  The 16-byte reads then start
// at any element; a quad that straddles an edge is read element by element from clamped places --
// of a k-contiguous operand only in the last k-tile, of the others only in the workgroups whose
// tile reaches past the edge.
// ---------------------------------------------------------------------------
template <bool TA, bool TB, int BM, int BN, bool ANY, int KG>
__global__ __launch_bounds__(256 * KG, KG == 4 ? 4 : 2) void gemm_f32_tiled_kernel(
    float const *__restrict__ A, float const *__restrict__ B, float *C, int M, int N, int K, int64_t lda,
    int64_t ldb, int64_t ldc, float const *__restrict__ bias, int act, int accumulate) {
  constexpr int BKT = 32;
  constexpr int TMW = BM / 64, TNW = BN / 64;  // 32-row / 32-column blocks per wave
  constexpr bool A_KC = !TA, B_KC = TB;     // reduction index contiguous in memory
  constexpr int A_CH = BM * BKT / 4 / 256, B_CH = BN * BKT / 4 / 256;  // 16-byte chunks per thread and tile
  constexpr int A_SP = 2 * BM + 4, B_SP = 2 * BN + 4;                  // pair-layout row strides
  constexpr int A_FLOATS = A_KC ? (BKT / 2) * A_SP : BKT * BM;
  constexpr int B_FLOATS = B_KC ? (BKT / 2) * B_SP : BKT * BN;
  __shared__ __attribute__((aligned(16))) float As_all[KG][2][A_FLOATS];
  __shared__ __attribute__((aligned(16))) float Bs_all[KG][2][B_FLOATS];
  int const group = KG > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8) : 0;
  auto &As = As_all[group];
  auto &Bs = Bs_all[group];
  int const t = threadIdx.x & 255, lane = t & 63, wave = t >> 6;
  int const h = lane >> 5, l32 = lane & 31;
  int const wm0 = (wave >> 1) * (BM / 2), wn0 = (wave & 1) * (BN / 2);
  int tm, tn;
  tile_coords(blockIdx.x, (M + BM - 1) / BM, (N + BN - 1) / BN, tm, tn);
  int const m0 = tm * BM, n0 = tn * BN;

  // Chunk i of this thread: (row, k quad) of a k-contiguous operand, (k row, row quad) otherwise.
  // Its address for k-tile 0 is kept and moved on by a constant per tile; only a tile that
  // reaches past K (the last one of a ragged reduction) computes clamped addresses afresh.
  constexpr int NCH = A_CH + B_CH;
  f32x4 rgs[2][NCH];  // k-tile kt travels in set kt % 2, two tiles ahead of its use
  float const *pg[NCH];
#pragma unroll
  for (int i = 0; i < A_CH; i++) {
    int const c = t + i * 256;
    pg[i] = A_KC ? A + (int64_t)min(m0 + c / 8, M - 1) * lda + 4 * (c % 8)
                 : A + (int64_t)(c / (BM / 4)) * lda + (ANY ? m0 + 4 * (c % (BM / 4)) : min(m0 + 4 * (c % (BM / 4)), M - 4));
  }
#pragma unroll
  for (int i = 0; i < B_CH; i++) {
    int const c = t + i * 256;
    pg[A_CH + i] = B_KC ? B + (int64_t)min(n0 + c / 8, N - 1) * ldb + 4 * (c % 8)
                        : B + (int64_t)(c / (BN / 4)) * ldb + (ANY ? n0 + 4 * (c % (BN / 4)) : min(n0 + 4 * (c % (BN / 4)), N - 4));
  }
  // Every group of waves takes as many k-tiles, from `first` on; past the reduction's end they are zeros.
  int const KT = ((K + BKT - 1) / BKT + KG - 1) / KG, first = group * KT;
  int64_t const step_a = A_KC ? BKT : (int64_t)BKT * lda, step_b = B_KC ? BKT : (int64_t)BKT * ldb;
  // load of chunk i of k-tile kt; pg[i] points at k-tile kt on entry and at kt + 1 on return
  auto gload_chunk = [&](int kt, int i, f32x4 (&rg)[NCH]) __attribute__((always_inline)) {
    int const k0 = (first + kt) * BKT;
    bool const is_a = i < A_CH;
    bool const kc = is_a ? A_KC : B_KC;
    // this chunk's tile reaches past the edge along the operand's contiguous index
    bool const straddles = ANY && (kc ? k0 + BKT > K : is_a ? m0 + BM > M : n0 + BN > N);  // uniform
    if (straddles) {
      int const c = t + (is_a ? i : i - A_CH) * 256;
      int const row = (is_a ? BM : BN) / 4;
      int const at = kc ? k0 + 4 * (c % 8) : (is_a ? m0 : n0) + 4 * (c % row);
      int const len = kc ? K : is_a ? M : N;
      // rows past K (of an operand lying [K][..]) are read from the last one
      float const *const p = kc || k0 + c / row < K ? pg[i] : pg[i] - (int64_t)(k0 + c / row - (K - 1)) * (is_a ? lda : ldb);
#pragma unroll
      for (int j = 0; j < 4; j++) rg[i][j] = p[min(j, len - 1 - at)];
    } else if (k0 + BKT <= K) {
      rg[i] = ANY ? __builtin_bit_cast(f32x4, load_raw_any(pg[i])) : *reinterpret_cast<f32x4 const *>(pg[i]);
    } else {
      int const c = t + (is_a ? i : i - A_CH) * 256;
      // how far this chunk's k lies past the last one it may read
      if (is_a ? A_KC : B_KC) {
        int const over = max(k0 + 4 * (c % 8) - (K - 4), 0);
        rg[i] = *reinterpret_cast<f32x4 const *>(pg[i] - over);
      } else {
        int const over = max(k0 + c / ((is_a ? BM : BN) / 4) - (K - 1), 0);
        float const *const p = pg[i] - (int64_t)over * (is_a ? lda : ldb);
        rg[i] = ANY ? __builtin_bit_cast(f32x4, load_raw_any(p)) : *reinterpret_cast<f32x4 const *>(p);
      }
    }
    pg[i] += is_a ? step_a : step_b;
  };
  auto gload = [&](int kt, f32x4 (&rg)[NCH]) {
#pragma unroll
    for (int i = 0; i < NCH; i++) gload_chunk(kt, i, rg);
  };
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  // chunk i of k-tile kt from its registers into buffer buf, k past the end zeroed
  auto lstore_chunk = [&](int buf, int kt, int i, f32x4 const (&rg)[NCH]) __attribute__((always_inline)) {
    f32x4 const zero = {0.0f, 0.0f, 0.0f, 0.0f};
    int const k0 = (first + kt) * BKT;
    bool const is_a = i < A_CH;
    int const c = t + (is_a ? i : i - A_CH) * 256;
    float *dst = is_a ? As[buf] : Bs[buf];
    int const SP = is_a ? A_SP : B_SP, R = is_a ? BM : BN;
    // (vector instructions between the MFMAs are not free: with two waves on a SIMD the masks
    // and selects of this function, applied to every tile, cost 5-10% of the matrix pipe's time.
    // The mask is for the one tile that reaches past K; which blocks are swapped is known per chunk.)
    bool const whole = k0 + BKT <= K;  // uniform
    if (is_a ? A_KC : B_KC) {
      int const row = c / 8, kq = c % 8;
      f32x4 v = rg[i];
      if (!whole) {
        asm volatile("" ::: "memory");  // a branch, not four selects on every tile
        if constexpr (ANY) {
#pragma unroll
          for (int j = 0; j < 4; j++) v[j] = k0 + 4 * kq + j < K ? v[j] : 0.0f;
        } else {
          v = k0 + 4 * kq < K ? v : zero;
        }
      }
      // odd 32-row blocks hold their k pairs swapped; row / 32 = chunk number (t / 8 < 32)
      bool const odd = (((is_a ? i : i - A_CH) & 1) != 0);
      *reinterpret_cast<f32x2 *>(&dst[(2 * kq) * SP + 2 * row]) = odd ? f32x2{v[1], v[0]} : f32x2{v[0], v[1]};
      *reinterpret_cast<f32x2 *>(&dst[(2 * kq + 1) * SP + 2 * row]) = odd ? f32x2{v[3], v[2]} : f32x2{v[2], v[3]};
    } else {
      int const k = c / (R / 4), rq = c % (R / 4);
      f32x4 v = rg[i];
      if (!whole) {
        asm volatile("" ::: "memory");
        v = k0 + k < K ? v : zero;
      }
      *reinterpret_cast<f32x4 *>(&dst[k * R + ((4 * rq) ^ ((k & 1) * 32))]) = v;
    }
  };
  // operand value of this lane for MFMA step kk (k = 2 kk + h) and its row
  auto frag_a = [&](int buf, int kk, int row) -> float {
    return A_KC ? As[buf][kk * A_SP + 2 * row + (h ^ ((row >> 5) & 1))] : As[buf][(2 * kk + h) * BM + (row ^ (h * 32))];
  };
  auto frag_b = [&](int buf, int kk, int row) -> float {
    return B_KC ? Bs[buf][kk * B_SP + 2 * row + (h ^ ((row >> 5) & 1))] : Bs[buf][(2 * kk + h) * BN + (row ^ (h * 32))];
  };

  f32x16 acc[TMW][TNW];
#pragma unroll
  for (int i = 0; i < TMW; i++)
#pragma unroll
    for (int j = 0; j < TNW; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;

  if constexpr (KG > 1) {
#pragma unroll
    for (int i = 0; i < NCH; i++) pg[i] += first * (i < A_CH ? step_a : step_b);
  }
  gload(0, rgs[0]);
  if (KT > 1) gload(1, rgs[1]);
#pragma unroll
  for (int i = 0; i < NCH; i++) lstore_chunk(0, 0, i, rgs[0]);
  __syncthreads();
  // One k-tile, kt, from buffer kt % 2.  AHEAD2: k-tile kt + 2 exists; its loads go out one per
  // step in the first NCH steps (a burst of them holds the wave, and with it its MFMAs, for as
  // long as the memory pipeline takes to accept them), into the register set that tile kt
  // travelled in.  AHEAD1: k-tile kt + 1
  // exists; it was asked for a tile ago and is written to the other buffer (which nobody reads
  // during this tile) one chunk per step in the last NCH steps, under the MFMAs.  A wave sits
  // at each MFMA until the pipe takes it, so whatever is placed between two of them costs
  // nothing as long as it is short; the fences keep it there.
  constexpr int KS = BKT / 2;
  static_assert(NCH <= KS, "one chunk per step");
  auto tile = [&](int kt, auto set_tag, auto ahead1_tag, auto ahead2_tag) {
    constexpr int SET = decltype(set_tag)::value;  // = kt % 2
    constexpr bool AHEAD1 = decltype(ahead1_tag)::value, AHEAD2 = decltype(ahead2_tag)::value;
    float af[2][TMW], bfv[2][TNW];
#pragma unroll
    for (int i = 0; i < TMW; i++) af[0][i] = frag_a(SET, 0, wm0 + i * 32 + l32);
#pragma unroll
    for (int j = 0; j < TNW; j++) bfv[0][j] = frag_b(SET, 0, wn0 + j * 32 + l32);
#pragma unroll
    for (int kk = 0; kk < KS; kk++) {
      int const c = kk & 1, nx = c ^ 1;
      // the next step's fragments are asked for before this step's MFMAs are issued: reads
      // issued behind them would start their round trip only when the last one has gone
      if (kk + 1 < KS) {
#pragma unroll
        for (int i = 0; i < TMW; i++) af[nx][i] = frag_a(SET, kk + 1, wm0 + i * 32 + l32);
#pragma unroll
        for (int j = 0; j < TNW; j++) bfv[nx][j] = frag_b(SET, kk + 1, wn0 + j * 32 + l32);
      }
      __builtin_amdgcn_sched_barrier(0);
      acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[c][0], bfv[c][0], acc[0][0], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (AHEAD2 && kk < NCH) gload_chunk(kt + 2, kk, rgs[SET]);
      if (AHEAD1 && kk >= KS - NCH) lstore_chunk(SET ^ 1, kt + 1, kk - (KS - NCH), rgs[SET ^ 1]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < TMW; i++)
#pragma unroll
        for (int j = 0; j < TNW; j++)
          if (i + j > 0) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[c][i], bfv[c][j], acc[i][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
  };
  using T0 = std::integral_constant<int, 0>;
  using T1 = std::integral_constant<int, 1>;
  int kt = 0;
  for (; kt + 3 < KT; kt += 2) {  // both tiles of the pair have two successors
    tile(kt, T0{}, std::true_type{}, std::true_type{});
    tile(kt + 1, T1{}, std::true_type{}, std::true_type{});
  }
  // the last one to three tiles (kt is even)
  if (kt + 2 < KT) {
    tile(kt, T0{}, std::true_type{}, std::true_type{});
    tile(kt + 1, T1{}, std::true_type{}, std::false_type{});
    tile(kt + 2, T0{}, std::false_type{}, std::false_type{});
  } else if (kt + 1 < KT) {
    tile(kt, T0{}, std::true_type{}, std::false_type{});
    tile(kt + 1, T1{}, std::false_type{}, std::false_type{});
  } else {
    tile(kt, T0{}, std::false_type{}, std::false_type{});
  }

  if constexpr (KG > 1) {  // the groups' sums meet in LDS
    static_assert((KG - 1) * 4 * TMW * TNW * 1024 <= KG * 2 * A_FLOATS, "they fit the tiles' room");
    float *const sums = &As_all[0][0][0];
    auto at = [&](int w, int i, int j, int g) {
      return reinterpret_cast<f32x4 *>(sums) + ((((w * 4 + wave) * TMW + i) * TNW + j) * 4 + g) * 64 + lane;
    };
#pragma unroll
    for (int i = 0; i < TMW; i++)
#pragma unroll
      for (int j = 0; j < TNW; j++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
          if (group > 0) *at(group - 1, i, j, g) = f32x4{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
        }
    __syncthreads();
    if (group > 0) return;
#pragma unroll
    for (int w = 0; w < KG - 1; w++)
#pragma unroll
      for (int i = 0; i < TMW; i++)
#pragma unroll
        for (int j = 0; j < TNW; j++)
#pragma unroll
          for (int g = 0; g < 4; g++) {
            f32x4 const x = *at(w, i, j, g);
#pragma unroll
            for (int e = 0; e < 4; e++) acc[i][j][4 * g + e] += x[e];
          }
  }
  // accumulator element r of lane l: row 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32 of its block
#pragma unroll
  for (int j = 0; j < TNW; j++) {
    int const n = n0 + wn0 + j * 32 + l32;
    if (n >= N) continue;
    float const bv = bias != nullptr ? bias[n] : 0.0f;
#pragma unroll
    for (int i = 0; i < TMW; i++) {
      int const mb = m0 + wm0 + i * 32 + 4 * h;
      float old[16];
      if (accumulate) {  // what C holds, all loads in flight together
#pragma unroll
        for (int r = 0; r < 16; r++) {
          int const m = min(mb + 8 * (r >> 2) + (r & 3), M - 1);
          old[r] = C[(int64_t)m * ldc + n];
        }
      }
#pragma unroll
      for (int r = 0; r < 16; r++) {
        int const m = mb + 8 * (r >> 2) + (r & 3);
        float v = apply_activation(acc[i][j][r] + bv, act);
        if (accumulate) v += old[r];
        if (m < M) C[(int64_t)m * ldc + n] = v;
      }
    }
  }
}

// Few outputs, or a long reduction over few: four waves a tile of 16 x 16 or 32 x 32, sixteen where the
// reduction is long (small_f32.h), where block tiles would leave most of the chip idle and walk the
// reduction alone ([25,1024] over 42 023: 1180 us with sixteen workgroups of 64 x 64; 138 x 640 over 640, a
// short sequence's projections: 20 us with thirty, 8-10 so).
template <bool TA, bool TB, int T, int WAVES, typename Store>
__device__ __forceinline__ void f32_small_tile(float const *A, float const *B, int M, int N, int K, int64_t lda, int64_t ldb,
                                               Store const &store) {
  __shared__ SmallShared<T, WAVES> sm;
  int const nbn = (N + T - 1) / T, tm = (int)blockIdx.x / nbn, tn = (int)blockIdx.x - tm * nbn;
  SmallOperand<!TA, FFK_ACT_NONE> const a = {A, nullptr, lda, 0};
  SmallOperand<TB, FFK_ACT_NONE> const b = {B, nullptr, ldb, 0};
  small_tile<T, WAVES, WAVES>(a, b, M, N, K, tm * T, tn * T, true, nullptr, 0, store, false, [](int, float) {}, sm);
}
__device__ __forceinline__ void f32_epilogue(float *C, int64_t ldc, float const *bias, int act, int accumulate, int m, int n,
                                             float v) {
  v = apply_activation(v + (bias != nullptr ? bias[n] : 0.0f), act);
  float *const to = C + (int64_t)m * ldc + n;
  *to = accumulate ? *to + v : v;
}

template <bool TA, bool TB, int T>
__global__ __launch_bounds__(256) void gemm_f32_small_kernel(float const *__restrict__ A, float const *__restrict__ B, float *C,
                                                             int M, int N, int K, int64_t lda, int64_t ldb, int64_t ldc,
                                                             float const *__restrict__ bias, int act, int accumulate) {
  f32_small_tile<TA, TB, T, 4>(A, B, M, N, K, lda, ldb,
                               [&](int m, int n, float v) { f32_epilogue(C, ldc, bias, act, accumulate, m, n, v); });
}

// partial != nullptr: workgroup row y takes the k's from y * k_per_split on and leaves its sums in
// partial[y][M][N], which gemm_f32_splits_kernel adds up.
template <bool TA, bool TB>
__global__ __launch_bounds__(1024) void gemm_f32_deep_kernel(float const *__restrict__ A, float const *__restrict__ B, float *C,
                                                             int M, int N, int K, int64_t lda, int64_t ldb, int64_t ldc,
                                                             float const *__restrict__ bias, int act, int accumulate,
                                                             float *partial, int k_per_split) {
  if (partial != nullptr) {
    int const k0 = (int)blockIdx.y * k_per_split;
    K = min(K - k0, k_per_split);
    A += TA ? (int64_t)k0 * lda : k0;
    B += TB ? k0 : (int64_t)k0 * ldb;
    partial += (int64_t)blockIdx.y * M * N;
  }
  f32_small_tile<TA, TB, 16, 16>(A, B, M, N, K, lda, ldb, [&](int m, int n, float v) {
    if (partial != nullptr) {
      partial[(int64_t)m * N + n] = v;
    } else {
      f32_epilogue(C, ldc, bias, act, accumulate, m, n, v);
    }
  });
}

__global__ __launch_bounds__(256) void gemm_f32_splits_kernel(float const *__restrict__ partial, float *C, int M, int N,
                                                              int64_t ldc, float const *__restrict__ bias, int act,
                                                              int accumulate, int splits) {
  int64_t const at = (int64_t)blockIdx.x * 256 + threadIdx.x, total = (int64_t)M * N;
  if (at >= total) return;
  int const m = (int)(at / N), n = (int)(at - (int64_t)m * N);
  float v = 0.0f;
  for (int s = 0; s < splits; s++) v += partial[s * total + at];
  f32_epilogue(C, ldc, bias, act, accumulate, m, n, v);
}

template <bool TA, bool TB, int BM, int BN, bool ANY, int KG>
static void launch_tiled(hipStream_t st, int M, int N, int K, float const *A, int64_t lda, float const *B, int64_t ldb,
                         float *C, int64_t ldc, GemmEpilogue const &ep) {
  if (describe_only("gemm_f32_tiled_kernel<%s,%s,%d,%d,%s,%d>", tf(TA), tf(TB), BM, BN, tf(ANY), KG)) return;
  gemm_f32_tiled_kernel<TA, TB, BM, BN, ANY, KG><<<(int)(ceil_div(M, BM) * ceil_div(N, BN)), 256 * KG, 0, st>>>(
      A, B, C, M, N, K, lda, ldb, ldc, static_cast<float const *>(ep.bias), ep.activation, ep.accumulate);
}

template <bool TA, bool TB>
static void pick_f32(hipStream_t st, int M, int N, int K, float const *A, int64_t lda, float const *B, int64_t ldb,
                     float *C, int64_t ldc, GemmEpilogue const &ep) {
  float const *const bias = static_cast<float const *>(ep.bias);
  // Tiles of sixteen waves, one round of two a CU at most: 200 x 200 over 3000 12 us, 16 on tiles of four waves, which
  // are ahead from one of them a CU on (300 x 300 over 4096 36 and 31, 512 x 512 55 and 48), but tests name these.
  if (K >= 2048 && ceil_div(M, 16) * ceil_div(N, 16) <= 2 * kNumCU) {
    // Two workgroups a CU: with scratch at hand, reductions of thousands are split over workgroups until
    // there are ([476, 58] over 40 305: 147 us with 120 workgroups,
    // 102 with 600 and the 5 of adding up; [128, 45] over 21 856: 72 and 14 + 7).
    int64_t const tiles = ceil_div(M, 16) * ceil_div(N, 16);
    int64_t const most = std::min<int64_t>(K / 1024, (int64_t)(ep.splitk_ws_bytes / sizeof(float)) / ((int64_t)M * N));
    int64_t const want = std::min<int64_t>(ceil_div(2 * kNumCU, tiles), most);
    if (describe_only("gemm_f32_deep_kernel<%s,%s>", tf(TA), tf(TB))) return;
    if (ep.splitk_ws != nullptr && want > 1) {
      int const per = (int)(ceil_div(ceil_div(K, want), 64) * 64), splits = (int)ceil_div(K, per);
      float *const partial = static_cast<float *>(ep.splitk_ws);
      gemm_f32_deep_kernel<TA, TB><<<dim3((unsigned)tiles, (unsigned)splits), 1024, 0, st>>>(
          A, B, C, M, N, K, lda, ldb, ldc, nullptr, FFK_ACT_NONE, 0, partial, per);
      gemm_f32_splits_kernel<<<(unsigned)ceil_div((int64_t)M * N, 256), 256, 0, st>>>(partial, C, M, N, ldc, bias, ep.activation,
                                                                                     ep.accumulate, splits);
      return;
    }
    gemm_f32_deep_kernel<TA, TB><<<(unsigned)tiles, 1024, 0, st>>>(A, B, C, M, N, K, lda, ldb, ldc, bias, ep.activation,
                                                                   ep.accumulate, nullptr, 0);
    return;
  }
  // The areas up to which the small Linear's forward keeps these tiles, four fifths of them where the reduction is
  // long: 64 x 64 tiles, one a CU at most, walk it alone (225 x 2048 over 6144 148 us, 92 so; 256 x 256 over 1095 29
  // and 6.5; 500 x 1000 over 1300 35 and 25; 320 x 1992 over 2688, past the line, 68 and 75), and so do the guarded
  // ones below (21 x 80 over 1344 84 and 6.0, 25 x 380 over 256 20 and 4.3).  (Short reductions stay on those, which
  // tests name: 32 x 128 over 64 8.2 us launch to launch, the small Linear's forward on these tiles 3.6.)
  int64_t const area = (int64_t)M * N;
  if (K >= (area < 128 * 128 ? 128 : 256) && M < (1 << 20) && N < (1 << 20)) {
    int const t = area <= 16 * 16 * 1024 ? 16 : 32;
    if (area <= 32 * 32 * (K <= 1024 ? 640 : 512)) {
      if (describe_only("gemm_f32_small_kernel<%s,%s,%d>", tf(TA), tf(TB), t)) return;
      auto kern = t == 16 ? gemm_f32_small_kernel<TA, TB, 16> : gemm_f32_small_kernel<TA, TB, 32>;
      kern<<<(unsigned)(ceil_div(M, t) * ceil_div(N, t)), 256, 0, st>>>(A, B, C, M, N, K, lda, ldb, ldc, bias, ep.activation,
                                                                        ep.accumulate);
      return;
    }
  }
  if ((int64_t)M * N < 128 * 128 || K < 4) {
    if (describe_only("gemm_f32_kernel<%s,%s>", tf(TA), tf(TB))) return;
    gemm_f32_kernel<TA, TB><<<(int)(ceil_div(M, 64) * ceil_div(N, 64)), 256, 0, st>>>(
        A, B, C, M, N, K, lda, ldb, ldc, static_cast<float const *>(ep.bias), ep.activation, ep.accumulate);
    return;
  }
  // 16-byte reads: aligned rows, and whole quads along whichever index is contiguous
  bool const quads = aligned16(A) && aligned16(B) && lda % 4 == 0 && ldb % 4 == 0 && (TA ? M : K) % 4 == 0 && (TB ? K : N) % 4 == 0 &&
                     M >= 4 && N >= 4;
  // 128 x 128 tiles when they give every CU two workgroups, 128 x 64 when those reach three quarters
  // of the CUs, 64 x 64 below and where half a 128-row tile would be empty.  And 64 x 64 where the CU with the most
  // of them has less to do than the one with the most of the others: the kernel is bound by the matrix pipe, so an
  // idle CU is lost (6144 x 512 over 4096, 384 tiles of 128 x 64 or 768 of 64 x 64 on 256 CUs, 263 -> 217 us; 3045 x
  // 1024 over 3072 202 -> 166; 1500 x 1500 over 1500 103 -> 83; where both have as much, 5% behind).
  auto busiest = [&](int bm, int bn) { return ceil_div(ceil_div(M, bm) * ceil_div(N, bn), kNumCU) * bm * bn; };
  int tile = M <= 64 ? 2 : ceil_div(M, 128) * ceil_div(N, 128) >= 2 * kNumCU ? 0 :
             ceil_div(M, 128) * ceil_div(N, 64) >= kNumCU * 3 / 4 ? 1 : 2;
  if (tile != 2 && busiest(64, 64) < 0.95 * (double)(tile == 0 ? busiest(128, 128) : busiest(128, 64))) tile = 2;
  // One workgroup a CU: two 64 x 64 tiles a CU become one of 128 x 64, and groups of waves split the reduction, so that
  // a SIMD has another wave's MFMAs while one waits for its fragments (4096 x 512 over 6144 250 -> 231 us, 1075 x 1024
  // over 3072 118 -> 104; 1024 x 1024 over 3045 73 -> 62 on two groups, 60 on four, over 752 22.3, 19.8 and 20.0, over
  // 300 12.3, 11.7 and 13.3, of 1030 x 520 over 200 9.5 and 9.8.  With more workgroups that is so as it is, and the
  // groups lose: 1866 x 3072 over 1024, 360 tiles of 128 x 64, 104 and 116.)  Not where one column of tiles reads A from
  // memory just once: half as many workgroups then have fewer reads under way (19253 x 54 over 2048 105 -> 117 us,
  // 24000 x 56 over 512 25 -> 29; of two columns, 9000 x 112 over 2048, 80 -> 77).
  int64_t const t64 = ceil_div(M, 64) * ceil_div(N, 64), t128x64 = ceil_div(M, 128) * ceil_div(N, 64);
  if (tile == 2 && M > 64 && N > 64 && t64 > kNumCU && t128x64 <= kNumCU) tile = 1;
  int const kg = K < 256 || (tile == 1 ? t128x64 : t64) > kNumCU ? 1 : tile == 2 && K >= 2048 ? 4 : 2;
#define FFK_F32(BM_, BN_, KG_)                                                              \
  do {                                                                                      \
    if (quads)                                                                              \
      launch_tiled<TA, TB, BM_, BN_, false, KG_>(st, M, N, K, A, lda, B, ldb, C, ldc, ep);  \
    else                                                                                    \
      launch_tiled<TA, TB, BM_, BN_, true, KG_>(st, M, N, K, A, lda, B, ldb, C, ldc, ep);   \
  } while (0)
  if (tile == 0) FFK_F32(128, 128, 1);
  else if (tile == 1 && kg == 2) FFK_F32(128, 64, 2);
  else if (tile == 1) FFK_F32(128, 64, 1);
  else if (kg == 4) FFK_F32(64, 64, 4);
  else if (kg == 2) FFK_F32(64, 64, 2);
  else FFK_F32(64, 64, 1);
#undef FFK_F32
}

hipError_t gemm_f32_launch(hipStream_t st, bool ta, bool tb, int M, int N, int K, float const *A, int64_t lda,
                           float const *B, int64_t ldb, float *C, int64_t ldc, GemmEpilogue const &ep) {
  if (!ta && !tb) pick_f32<false, false>(st, M, N, K, A, lda, B, ldb, C, ldc, ep);
  else if (!ta && tb) pick_f32<false, true>(st, M, N, K, A, lda, B, ldb, C, ldc, ep);
  else if (ta && !tb) pick_f32<true, false>(st, M, N, K, A, lda, B, ldb, C, ldc, ep);
  else pick_f32<true, true>(st, M, N, K, A, lda, B, ldb, C, ldc, ep);
  return tl_name_sink != nullptr ? hipSuccess : hipGetLastError();
}

}  // namespace ffk
