// GEMM kernels for gfx950 behind Linear and the attention projections.
//
//  * bf16 (gemm_bf16.h): LDS-tiled, pipelined MFMA kernels (v_mfma_f32_32x32x16_bf16,
//    fp32 accumulators, one rounding at the store).  Operands whose reduction
//    dimension is not contiguous in memory are staged into LDS as they lie in
//    memory and read back with the transposing LDS load (ds_read_b64_tr_b16),
//    so all four transpose variants run on the same pipeline.  Operands that cannot
//    be read 16 aligned bytes at a time run on a register-staged kernel, products of
//    very few elements on a plain one-thread-per-output kernel.
//  * fp32: MFMA v_mfma_f32_32x32x2f32 kernels, tiled for operands readable 16 bytes at a
//    time, bounds-checked for the others.
//
// These replace the cublasGemmEx calls of the reference
// (lib/kernels/src/cuda/ops/linear_kernels.cu:143,163,249,298,321).
#include "lds_dma.h"
#include "gemm.h"
#include "colreduce.h"
#include "gemm_bf16.h"
#include <stdlib.h>

namespace ffk {

// instantiated in gemm_nn.hip, gemm_nt.hip, gemm_tn.hip, gemm_tt.hip
#define FFK_EXTERN_BF16(TA_, TB_)                                                                                       \
  extern template hipError_t pick_bf16<TA_, TB_>(hipStream_t, bf16 const *, bf16 const *, bf16 *, int, int, int,        \
                                                 int64_t, int64_t, int64_t, GemmEpilogue const &, bool);                \
  extern template hipError_t launch_pipe_pair<TA_, TB_>(hipStream_t, GemmProblem const &, GemmProblem const &, int, bool)
FFK_EXTERN_BF16(false, false);
FFK_EXTERN_BF16(false, true);
FFK_EXTERN_BF16(true, false);
FFK_EXTERN_BF16(true, true);
#undef FFK_EXTERN_BF16

size_t gemm_splitk_workspace_bytes(int dtype, int64_t M, int64_t N, int64_t K) {
  if (dtype != FFK_BF16 || M % 128 != 0 || N % 128 != 0) return 0;
  int const s = splitk_splits(M, N, K, ~(size_t)0);
  return s > 1 ? (size_t)s * (size_t)(M * N) * sizeof(float) : 0;
}

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
// fp32 MFMA kernel for operands that can be read 16 bytes at a time: 128 x BN
// block tile (BN = 128 or 64), 2 x 2 waves of 64 x BN/2, reduction tiles of 32.
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
// without padding.  Every element's products are added in ascending k, two per
// MFMA, as in gemm_f32_kernel: the two kernels give the same bits.
// Rows and columns past the edge are read from the last valid ones and never
// stored; k past the end is zeroed when the tile is written to LDS.
// ---------------------------------------------------------------------------
template <bool TA, bool TB, int BN>
__global__ __launch_bounds__(256, 2) void gemm_f32_tiled_kernel(
    float const *__restrict__ A, float const *__restrict__ B, float *C, int M, int N, int K, int64_t lda,
    int64_t ldb, int64_t ldc, float const *__restrict__ bias, int act, int accumulate) {
  constexpr int BM = 128, BKT = 32;
  constexpr int TNW = BN / 64;              // 32-column blocks per wave
  constexpr bool A_KC = !TA, B_KC = TB;     // reduction index contiguous in memory
  constexpr int A_CH = BM * BKT / 4 / 256, B_CH = BN * BKT / 4 / 256;  // 16-byte chunks per thread and tile
  constexpr int A_SP = 2 * BM + 4, B_SP = 2 * BN + 4;                  // pair-layout row strides
  constexpr int A_FLOATS = A_KC ? (BKT / 2) * A_SP : BKT * BM;
  constexpr int B_FLOATS = B_KC ? (BKT / 2) * B_SP : BKT * BN;
  __shared__ __attribute__((aligned(16))) float As[2][A_FLOATS];
  __shared__ __attribute__((aligned(16))) float Bs[2][B_FLOATS];
  int const t = threadIdx.x, lane = t & 63, wave = t >> 6;
  int const h = lane >> 5, l32 = lane & 31;
  int const wm0 = (wave >> 1) * 64, wn0 = (wave & 1) * (BN / 2);
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
                 : A + (int64_t)(c / (BM / 4)) * lda + min(m0 + 4 * (c % (BM / 4)), M - 4);
  }
#pragma unroll
  for (int i = 0; i < B_CH; i++) {
    int const c = t + i * 256;
    pg[A_CH + i] = B_KC ? B + (int64_t)min(n0 + c / 8, N - 1) * ldb + 4 * (c % 8)
                        : B + (int64_t)(c / (BN / 4)) * ldb + min(n0 + 4 * (c % (BN / 4)), N - 4);
  }
  int64_t const step_a = A_KC ? BKT : (int64_t)BKT * lda, step_b = B_KC ? BKT : (int64_t)BKT * ldb;
  // load of chunk i of k-tile kt; pg[i] points at k-tile kt on entry and at kt + 1 on return
  auto gload_chunk = [&](int kt, int i, f32x4 (&rg)[NCH]) __attribute__((always_inline)) {
    int const k0 = kt * BKT;
    bool const is_a = i < A_CH;
    if (k0 + BKT <= K) {
      rg[i] = *reinterpret_cast<f32x4 const *>(pg[i]);
    } else {
      int const c = t + (is_a ? i : i - A_CH) * 256;
      // how far this chunk's k lies past the last one it may read
      if (is_a ? A_KC : B_KC) {
        int const over = max(k0 + 4 * (c % 8) - (K - 4), 0);
        rg[i] = *reinterpret_cast<f32x4 const *>(pg[i] - over);
      } else {
        int const over = max(k0 + c / ((is_a ? BM : BN) / 4) - (K - 1), 0);
        rg[i] = *reinterpret_cast<f32x4 const *>(pg[i] - (int64_t)over * (is_a ? lda : ldb));
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
    int const k0 = kt * BKT;
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
        v = k0 + 4 * kq < K ? v : zero;
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

  f32x16 acc[2][TNW];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < TNW; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;

  int const KT = (K + BKT - 1) / BKT;
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
    float af[2][2], bfv[2][TNW];
#pragma unroll
    for (int i = 0; i < 2; i++) af[0][i] = frag_a(SET, 0, wm0 + i * 32 + l32);
#pragma unroll
    for (int j = 0; j < TNW; j++) bfv[0][j] = frag_b(SET, 0, wn0 + j * 32 + l32);
#pragma unroll
    for (int kk = 0; kk < KS; kk++) {
      int const c = kk & 1, nx = c ^ 1;
      // the next step's fragments are asked for before this step's MFMAs are issued: reads
      // issued behind them would start their round trip only when the last one has gone
      if (kk + 1 < KS) {
#pragma unroll
        for (int i = 0; i < 2; i++) af[nx][i] = frag_a(SET, kk + 1, wm0 + i * 32 + l32);
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
      for (int i = 0; i < 2; i++)
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

  // accumulator element r of lane l: row 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32 of its block
#pragma unroll
  for (int j = 0; j < TNW; j++) {
    int const n = n0 + wn0 + j * 32 + l32;
    if (n >= N) continue;
    float const bv = bias != nullptr ? bias[n] : 0.0f;
#pragma unroll
    for (int i = 0; i < 2; i++) {
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

// ---------------------------------------------------------------------------
// Plain kernel for bf16 shapes the tiled kernel cannot take.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void gemm_bf16_plain_kernel(
    bf16 const *__restrict__ A, bf16 const *__restrict__ B, bf16 *C, int M,
    int N, int K, int64_t lda, int64_t ldb, int64_t ldc, int ta, int tb,
    bf16 const *__restrict__ bias, int act, int accumulate) {
  int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (int64_t)M * N) return;
  int m = (int)(idx / N), n = (int)(idx % N);
  float acc = 0.0f;
  for (int k = 0; k < K; k++) {
    float a = VecIO<bf16>::load1(ta ? A + (int64_t)k * lda + m : A + (int64_t)m * lda + k);
    float b = VecIO<bf16>::load1(tb ? B + (int64_t)n * ldb + k : B + (int64_t)k * ldb + n);
    acc += a * b;
  }
  if (bias != nullptr) acc += VecIO<bf16>::load1(bias + n);
  acc = apply_activation(acc, act);
  bf16 *dst = C + (int64_t)m * ldc + n;
  if (accumulate) acc += VecIO<bf16>::load1(dst);
  VecIO<bf16>::store1(dst, acc);
}

// ---------------------------------------------------------------------------
// Column sums (bias gradient): out[n] (+)= sum_m X[m,n]
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void colsum_partial_kernel(
    T const *__restrict__ X, int64_t ldx, int M, int N, int rows_per_split,
    float *__restrict__ partials) {
  __shared__ float red[4][64];
  int const cx = threadIdx.x & 63;
  int const ry = threadIdx.x >> 6;
  int const n = blockIdx.x * 64 + cx;
  int const r0 = blockIdx.y * rows_per_split;
  int const r1 = min(M, r0 + rows_per_split);
  float s = 0.0f;
  if (n < N) {
    for (int m = r0 + ry; m < r1; m += 4) {
      s += VecIO<T>::load1(X + (int64_t)m * ldx + n);
    }
  }
  red[ry][cx] = s;
  __syncthreads();
  if (ry == 0 && n < N) {
    partials[(int64_t)blockIdx.y * N + n] =
        red[0][cx] + red[1][cx] + red[2][cx] + red[3][cx];
  }
}

// Vectorised first pass: a thread reads 16 bytes (8 bf16 / 4 fp32 columns) of
// kColsumRowsPerLane rows, all loads independent; 64 threads span the columns,
// the 4 row lanes of the workgroup meet in LDS.

// DROP: X is the gradient of a dropout's output; what is summed is the
// dropout's backward of it, rounded as stored, which is also written to G
// (dense, ldx == N: a lane's V elements are a Philox block or half of one).
template <typename T, bool DROP>
__global__ __launch_bounds__(256) void colsum_partial_vec_kernel(
    T const *__restrict__ X, int64_t ldx, int M, int N, int rows_per_split,
    float *__restrict__ partials, T *__restrict__ G, DropoutParams drop) {
  constexpr int V = VecIO<T>::kVec;
  __shared__ float red[4][64][V + 1];
  int const cx = threadIdx.x & 63;
  int const ry = threadIdx.x >> 6;
  int const n = (blockIdx.x * 64 + cx) * V;
  int const r0 = blockIdx.y * rows_per_split;
  int const r1 = min(M, r0 + rows_per_split);
  float s[V];
#pragma unroll
  for (int e = 0; e < V; e++) s[e] = 0.0f;
  if (n < N) {
    for (int m0 = r0 + ry * kColsumRowsPerLane; m0 < r1; m0 += kColsumRowsPerBlock) {
      float v[kColsumRowsPerLane][V];
#pragma unroll
      for (int i = 0; i < kColsumRowsPerLane; i++) {
        int const m = min(m0 + i, r1 - 1);  // clamped rows are masked below
        VecIO<T>::load_stream(X + (int64_t)m * ldx + n, v[i]);
      }
#pragma unroll
      for (int i = 0; i < kColsumRowsPerLane; i++) {
        if (m0 + i < r1) {
          if constexpr (DROP) {
            uint64_t const e0 = drop.offset + (uint64_t)(m0 + i) * (uint64_t)N + (uint64_t)n;
            uint32_t w[4];
            philox4x32_10(e0 >> 3, drop.key, w);
            if (V == 4 && (e0 & 4)) {  // upper half of the block
              w[0] = w[2];
              w[1] = w[3];
            }
#pragma unroll
            for (int e = 0; e < V; e++) v[i][e] = storage_round<T>(keep(w, e, drop) ? v[i][e] * drop.scale : 0.0f);
            VecIO<T>::store(G + (int64_t)(m0 + i) * ldx + n, v[i]);
          }
#pragma unroll
          for (int e = 0; e < V; e++) s[e] += v[i][e];
        }
      }
    }
  }
#pragma unroll
  for (int e = 0; e < V; e++) red[ry][cx][e] = s[e];
  __syncthreads();
  if (ry == 0 && n < N) {
#pragma unroll
    for (int e = 0; e < V; e++) {
      partials[(int64_t)blockIdx.y * N + n + e] =
          (red[0][cx][e] + red[1][cx][e]) + (red[2][cx][e] + red[3][cx][e]);
    }
  }
}

static int colsum_splits(int64_t M) {
  int64_t s = ceil_div(M, kColsumRowsPerBlock);
  return (int)(s < 1 ? 1 : (s > 256 ? 256 : s));
}

// Rows that one partial sum of the vector column-sum kernel covers.
static int64_t colsum_rows_per_split(int64_t M) {
  int64_t const rows = ceil_div(M, (int64_t)colsum_splits(M));
  return ceil_div(rows, (int64_t)kColsumRowsPerBlock) * kColsumRowsPerBlock;
}

int colsum_finish(hipStream_t st, int dtype, float const *partials, int64_t M, int64_t N, void *out,
                  bool accumulate) {
  FFK_REQUIRE(dtype == FFK_BF16 && M % kColsumRowsPerBlock == 0 && colsum_rows_per_split(M) == kColsumRowsPerBlock,
              "colsum_finish: partials of this shape do not come from a GEMM tail");
  FFK_HIP(colreduce_launch<bf16>(st, partials, (int)(M / kColsumRowsPerBlock), (int)N, (int)N,
                                 static_cast<bf16 *>(out), nullptr, accumulate));
  return FFK_OK;
}

int64_t colsum_partials_elems(int64_t M, int64_t N) {
  return (int64_t)colsum_splits(M) * N;
}

// dropped != nullptr: the sums are taken over dropout_backward(X), which is
// written to dropped; vector shapes only (FFK_ERR_UNSUPPORTED otherwise, before
// any launch).
template <typename T>
static int colsum_typed(hipStream_t st, T const *X, int64_t ldx, int64_t M,
                        int64_t N, T *out, bool accumulate, float *partials,
                        T *dropped = nullptr, DropoutParams const *drop = nullptr) {
  constexpr int V = VecIO<T>::kVec;
  int const splits = colsum_splits(M);
  int rows_per_split = (int)ceil_div(M, splits);
  bool const vec = (N % V == 0) && (ldx % V == 0) && aligned16(X);
  if (dropped != nullptr) {
    if (!vec || ldx != N || !aligned16(dropped) || (drop->offset & 7) != 0 || M >= (1ll << 31) || N >= (1ll << 31)) {
      return FFK_ERR_UNSUPPORTED;
    }
    rows_per_split = (int)(ceil_div(rows_per_split, kColsumRowsPerBlock) * kColsumRowsPerBlock);
    int const used = (int)ceil_div(M, rows_per_split);
    dim3 grid((unsigned)ceil_div(N, 64 * V), (unsigned)used);
    colsum_partial_vec_kernel<T, true><<<grid, 256, 0, st>>>(X, ldx, (int)M, (int)N, rows_per_split, partials,
                                                            dropped, *drop);
    FFK_CHECK_LAUNCH();
    FFK_HIP(colreduce_launch<T>(st, partials, used, (int)N, (int)N, out, nullptr, accumulate));
    return FFK_OK;
  }
  if (vec) {
    // whole row blocks per split so that only the last split has a ragged end
    rows_per_split = (int)(ceil_div(rows_per_split, kColsumRowsPerBlock) * kColsumRowsPerBlock);
    int const used = (int)ceil_div(M, rows_per_split);
    dim3 grid((unsigned)ceil_div(N, 64 * V), (unsigned)used);
    colsum_partial_vec_kernel<T, false><<<grid, 256, 0, st>>>(X, ldx, (int)M, (int)N, rows_per_split, partials,
                                                             nullptr, DropoutParams{});
    FFK_CHECK_LAUNCH();
    FFK_HIP(colreduce_launch<T>(st, partials, used, (int)N, (int)N, out, nullptr, accumulate));
    return FFK_OK;
  }
  dim3 grid((unsigned)ceil_div(N, 64), (unsigned)splits);
  colsum_partial_kernel<T><<<grid, 256, 0, st>>>(X, ldx, (int)M, (int)N, rows_per_split, partials);
  FFK_CHECK_LAUNCH();
  FFK_HIP(colreduce_launch<T>(st, partials, splits, (int)N, (int)N, out, nullptr, accumulate));
  return FFK_OK;
}

int colsum_dispatch(hipStream_t st, int dtype, void const *X, int64_t ldx,
                    int64_t M, int64_t N, void *out, bool accumulate,
                    float *partials) {
  FFK_REQUIRE(partials != nullptr, "colsum: partials scratch is NULL");
  if (dtype == FFK_FLOAT) {
    return colsum_typed<float>(st, static_cast<float const *>(X), ldx, M, N,
                               static_cast<float *>(out), accumulate, partials);
  }
  if (dtype == FFK_BF16) {
    return colsum_typed<bf16>(st, static_cast<bf16 const *>(X), ldx, M, N,
                              static_cast<bf16 *>(out), accumulate, partials);
  }
  return fail(FFK_ERR_UNSUPPORTED, "colsum: dtype %d not supported", dtype);
}

int dropout_backward_colsum(hipStream_t st, int dtype, void const *dy, void *dx, int64_t M, int64_t N,
                            void *colsum, bool accumulate, float *partials, DropoutParams const &drop) {
  FFK_REQUIRE(dy && dx && colsum && partials, "dropout_backward_colsum: NULL operand");
  FFK_REQUIRE(M > 0 && N > 0, "dropout_backward_colsum: non-positive dimension");
  if (dtype == FFK_FLOAT) {
    return colsum_typed<float>(st, static_cast<float const *>(dy), N, M, N, static_cast<float *>(colsum),
                               accumulate, partials, static_cast<float *>(dx), &drop);
  }
  if (dtype == FFK_BF16) {
    return colsum_typed<bf16>(st, static_cast<bf16 const *>(dy), N, M, N, static_cast<bf16 *>(colsum),
                              accumulate, partials, static_cast<bf16 *>(dx), &drop);
  }
  return FFK_ERR_UNSUPPORTED;
}

static bool pair_member_ok(bool ta, bool tb, GemmProblem const &p, int64_t K) {
  if (p.M <= 0 || p.N <= 0 || p.M % 128 != 0 || p.N % 128 != 0 || !p.A || !p.B || !p.C) return false;
  if (p.M >= (1ll << 31) || p.N >= (1ll << 31)) return false;
  if (p.lda < (ta ? p.M : K) || p.ldb < (tb ? K : p.N) || p.ldc < p.N) return false;
  bool const vec_ok = (p.lda % 8 == 0) && (p.ldb % 8 == 0) && aligned16(p.A) && aligned16(p.B);
  GemmEpilogue none;
  return vec_ok && pipe_tile_for(static_cast<bf16 const *>(p.C), (int)p.M, (int)p.N, (int)K, p.lda, p.ldb, p.ldc, none,
                                 128) == 128;
}

bool gemm_pair_supported(int dtype, bool ta, bool tb, int64_t K, GemmProblem const &p0, GemmProblem const &p1) {
  if (dtype != FFK_BF16 || K <= 0 || K % 64 != 0 || K >= (1ll << 31) || gemm_variant_override() != 0) return false;
  if (!pair_member_ok(ta, tb, p0, K) || !pair_member_ok(ta, tb, p1, K)) return false;
  // worth it when neither problem fills the chip on its own and the two together come closer
  int64_t const t0 = (p0.M / 128) * (p0.N / 128), t1 = (p1.M / 128) * (p1.N / 128);
  return t0 < 2 * kNumCU && t1 < 2 * kNumCU && t0 + t1 >= kNumCU / 2;
}

int gemm_dispatch_pair(hipStream_t st, int dtype, bool ta, bool tb, int64_t K, GemmProblem const &p0,
                       GemmProblem const &p1, bool accumulate) {
  FFK_REQUIRE(gemm_pair_supported(dtype, ta, tb, K, p0, p1),
              "gemm: these two problems do not run as one launch (ask gemm_pair_supported first)");
  hipError_t e;
  if (!ta && !tb) e = launch_pipe_pair<false, false>(st, p0, p1, (int)K, accumulate);
  else if (!ta && tb) e = launch_pipe_pair<false, true>(st, p0, p1, (int)K, accumulate);
  else if (ta && !tb) e = launch_pipe_pair<true, false>(st, p0, p1, (int)K, accumulate);
  else e = launch_pipe_pair<true, true>(st, p0, p1, (int)K, accumulate);
  FFK_HIP(e);
  return FFK_OK;
}

bool gemm_tail_supported(int dtype, bool ta, bool tb, int64_t M, int64_t N, int64_t K,
                         void const *A, int64_t lda, void const *B, int64_t ldb,
                         void const *C, int64_t ldc, GemmEpilogue const &ep) {
  if (dtype != FFK_BF16 || ta || ep.accumulate || ldc != N || M <= 0 || N <= 0 || K <= 0) return false;
  if (M >= (1ll << 31) || N >= (1ll << 31) || K >= (1ll << 31)) return false;
  if ((ep.tail_dropout.offset & 7) != 0) return false;
  if (ep.tail == GemmEpilogue::kTailGeluDropout) {
    if (!tb || ep.tail_out == nullptr || !aligned16(ep.tail_out)) return false;
  } else if (ep.tail == GemmEpilogue::kTailDropoutGeluGrad) {
    if (tb || ep.tail_in == nullptr || !aligned16(ep.tail_in)) return false;
    if (ep.tail_colsum_partials != nullptr && colsum_rows_per_split(M) != kColsumRowsPerBlock) return false;
  } else if (ep.tail == GemmEpilogue::kTailDropoutAdd) {
    if (!tb || ep.tail_in == nullptr || !aligned16(ep.tail_in)) return false;
  } else {
    return false;
  }
  bool const vec_ok = (K % 8 == 0) && (lda % 8 == 0) && (ldb % 8 == 0) && aligned16(A) && aligned16(B) &&
                      (tb || N % 8 == 0);
  return vec_ok && pipe_tile_for(static_cast<bf16 const *>(C), (int)M, (int)N, (int)K, lda, ldb, ldc, ep,
                                 gemm_variant_override()) != 0;
}

int gemm_dispatch(hipStream_t st, int dtype, bool ta, bool tb, int64_t M,
                  int64_t N, int64_t K, void const *A, int64_t lda,
                  void const *B, int64_t ldb, void *C, int64_t ldc,
                  GemmEpilogue const &ep) {
  FFK_REQUIRE(M >= 0 && N >= 0 && K >= 0, "gemm: negative dimension");
  if (M == 0 || N == 0) return FFK_OK;
  FFK_REQUIRE(A && B && C, "gemm: NULL operand");
  FFK_REQUIRE(M < (1ll << 31) && N < (1ll << 31) && K < (1ll << 31),
              "gemm: dimension exceeds 2^31");
  FFK_REQUIRE(lda >= (ta ? M : K) && ldb >= (tb ? K : N) && ldc >= N,
              "gemm: leading dimension smaller than the row length");
  hipError_t e;
  if (dtype == FFK_FLOAT) {
    FFK_REQUIRE(ep.tail == GemmEpilogue::kTailNone, "gemm: fused tails exist for bf16 only");
    float const *a = static_cast<float const *>(A);
    float const *b = static_cast<float const *>(B);
    float *c = static_cast<float *>(C);
    float const *bias = static_cast<float const *>(ep.bias);
    // 16-byte reads: aligned rows, and whole quads along whichever index is contiguous
    bool const tiled = aligned16(A) && aligned16(B) && lda % 4 == 0 && ldb % 4 == 0 && K >= 4 &&
                       (ta ? M % 4 == 0 && M >= 4 : K % 4 == 0) && (tb ? K % 4 == 0 : N % 4 == 0 && N >= 4) &&
                       M * N >= 128 * 128;
    if (tiled) {
      // 128 x 128 tiles when they give every CU two workgroups, 128 x 64 otherwise
      bool const wide = ceil_div(M, 128) * ceil_div(N, 128) >= 2 * kNumCU;
      int const tblocks = (int)(ceil_div(M, 128) * ceil_div(N, wide ? 128 : 64));
      if (describe_only("gemm_f32_tiled_kernel<%s,%s,%d>", tf(ta), tf(tb), wide ? 128 : 64)) return FFK_OK;
#define FFK_LAUNCH_F32T(TA_, TB_)                                              \
  do {                                                                         \
    if (wide)                                                                  \
      gemm_f32_tiled_kernel<TA_, TB_, 128><<<tblocks, 256, 0, st>>>(           \
          a, b, c, (int)M, (int)N, (int)K, lda, ldb, ldc, bias, ep.activation, ep.accumulate); \
    else                                                                       \
      gemm_f32_tiled_kernel<TA_, TB_, 64><<<tblocks, 256, 0, st>>>(            \
          a, b, c, (int)M, (int)N, (int)K, lda, ldb, ldc, bias, ep.activation, ep.accumulate); \
  } while (0)
      if (!ta && !tb) FFK_LAUNCH_F32T(false, false);
      else if (!ta && tb) FFK_LAUNCH_F32T(false, true);
      else if (ta && !tb) FFK_LAUNCH_F32T(true, false);
      else FFK_LAUNCH_F32T(true, true);
#undef FFK_LAUNCH_F32T
      FFK_CHECK_LAUNCH();
      return FFK_OK;
    }
    int const blocks = (int)(ceil_div(M, 64) * ceil_div(N, 64));
#define FFK_LAUNCH_F32(TA_, TB_)                                               \
  gemm_f32_kernel<TA_, TB_><<<blocks, 256, 0, st>>>(                           \
      a, b, c, (int)M, (int)N, (int)K, lda, ldb, ldc, bias, ep.activation,     \
      ep.accumulate)
    if (describe_only("gemm_f32_kernel<%s,%s>", tf(ta), tf(tb))) return FFK_OK;
    if (!ta && !tb) FFK_LAUNCH_F32(false, false);
    else if (!ta && tb) FFK_LAUNCH_F32(false, true);
    else if (ta && !tb) FFK_LAUNCH_F32(true, false);
    else FFK_LAUNCH_F32(true, true);
#undef FFK_LAUNCH_F32
    e = hipGetLastError();
  } else if (dtype == FFK_BF16) {
    FFK_REQUIRE(ep.tail == GemmEpilogue::kTailNone ||
                    gemm_tail_supported(dtype, ta, tb, M, N, K, A, lda, B, ldb, C, ldc, ep),
                "gemm: this shape has no fused tail (ask gemm_tail_supported first)");
    bf16 const *a = static_cast<bf16 const *>(A);
    bf16 const *b = static_cast<bf16 const *>(B);
    bf16 *c = static_cast<bf16 *>(C);
    // 16-byte chunks: the contiguous extent of each operand (K, or M / N) must be a multiple of 8
    // elements, rows 16-byte aligned.
    bool vec_ok = (ta ? M % 8 == 0 : K % 8 == 0) && (tb ? K % 8 == 0 : N % 8 == 0) && (lda % 8 == 0) &&
                  (ldb % 8 == 0) && aligned16(A) && aligned16(B) && K > 0;
    // Operands that are not: the register-staged kernel, but for products of so few elements that
    // one thread an output is over as soon.
    if (!vec_ok && (K == 0 || M * N * K < (1 << 21))) {
      int64_t total = M * N;
      if (describe_only("gemm_bf16_plain_kernel")) return FFK_OK;
      gemm_bf16_plain_kernel<<<(unsigned)ceil_div(total, 256), 256, 0, st>>>(
          a, b, c, (int)M, (int)N, (int)K, lda, ldb, ldc, ta, tb,
          static_cast<bf16 const *>(ep.bias), ep.activation, ep.accumulate);
      e = hipGetLastError();
    } else if (!ta && !tb) {
      e = pick_bf16<false, false>(st, a, b, c, (int)M, (int)N, (int)K, lda, ldb, ldc, ep, vec_ok);
    } else if (!ta && tb) {
      e = pick_bf16<false, true>(st, a, b, c, (int)M, (int)N, (int)K, lda, ldb, ldc, ep, vec_ok);
    } else if (ta && !tb) {
      e = pick_bf16<true, false>(st, a, b, c, (int)M, (int)N, (int)K, lda, ldb, ldc, ep, vec_ok);
    } else {
      e = pick_bf16<true, true>(st, a, b, c, (int)M, (int)N, (int)K, lda, ldb, ldc, ep, vec_ok);
    }
  } else {
    return fail(FFK_ERR_UNSUPPORTED, "gemm: dtype %d not supported", dtype);
  }
  FFK_HIP(e);
  return FFK_OK;
}

}  // namespace ffk

using namespace ffk;

extern "C" int ffk_gemm_kernel_name(int dtype, int trans_a, int trans_b, int64_t M, int64_t N, int64_t K,
                                    int has_bias, int activation, char *name, size_t name_bytes) {
  FFK_REQUIRE(name != nullptr && name_bytes > 0, "gemm_kernel_name: no room for the name");
  FFK_REQUIRE(M > 0 && N > 0 && K > 0, "gemm_kernel_name: non-positive dimension");
  name[0] = 0;
  // dense, 16-byte aligned operands: the addresses only have to pass the alignment checks,
  // nothing is launched while the sink is set
  void *const somewhere = reinterpret_cast<void *>(uintptr_t(1) << 20);
  GemmEpilogue ep;
  ep.bias = has_bias ? somewhere : nullptr;
  ep.activation = activation;
  tl_name_sink = name;
  tl_name_sink_bytes = name_bytes;
  int const rc = gemm_dispatch(nullptr, dtype, trans_a != 0, trans_b != 0, M, N, K, somewhere, trans_a ? M : K,
                               somewhere, trans_b ? K : N, somewhere, N, ep);
  tl_name_sink = nullptr;
  tl_name_sink_bytes = 0;
  return rc;
}

extern "C" int ffk_gemm(ffk_stream_t stream, int dtype, int trans_a,
                        int trans_b, int64_t M, int64_t N, int64_t K,
                        void const *A, void const *B, void *C, int accumulate) {
  GemmEpilogue ep;
  ep.accumulate = accumulate != 0;
  return gemm_dispatch(as_stream(stream), dtype, trans_a != 0, trans_b != 0, M,
                       N, K, A, trans_a ? M : K, B, trans_b ? K : N, C, N, ep);
}
