// GEMM kernels for gfx950 behind Linear and the attention projections.
//
//  * bf16 (gemm_bf16.h): LDS-tiled, pipelined MFMA kernels (v_mfma_f32_32x32x16_bf16,
//    fp32 accumulators, one rounding at the store).  Operands whose reduction
//    dimension is not contiguous in memory are staged into LDS as they lie in
//    memory and read back with the transposing LDS load (ds_read_b64_tr_b16),
//    so all four transpose variants run on the same pipeline.  Operands that cannot
//    be read 16 aligned bytes at a time run on a register-staged kernel, products of
//    very few elements on a plain one-thread-per-output kernel.
//  * fp32 (gemm_f32.hip): MFMA v_mfma_f32_32x32x2f32 kernels.
//
// These replace the cublasGemmEx calls of the reference
// (lib/kernels/src/cuda/ops/linear_kernels.cu:143,163,249,298,321).
#include "lds_dma.h"
#include "gemm.h"
#include "colreduce.h"
#include "gemm_bf16.h"
#include <stdlib.h>

namespace ffk {

// gemm_f32.hip
hipError_t gemm_f32_launch(hipStream_t st, bool ta, bool tb, int M, int N, int K, float const *A, int64_t lda,
                           float const *B, int64_t ldb, float *C, int64_t ldc, GemmEpilogue const &ep);

// instantiated in gemm_nn.hip, gemm_nt.hip, gemm_tn.hip, gemm_tt.hip
#define FFK_EXTERN_BF16(TA_, TB_)                                                                                       \
  extern template hipError_t pick_bf16<TA_, TB_>(hipStream_t, bf16 const *, bf16 const *, bf16 *, int, int, int,        \
                                                 int64_t, int64_t, int64_t, GemmEpilogue const &, bool)
FFK_EXTERN_BF16(false, false);
FFK_EXTERN_BF16(false, true);
FFK_EXTERN_BF16(true, false);
FFK_EXTERN_BF16(true, true);
#undef FFK_EXTERN_BF16
extern template hipError_t pick_bf16_tail<false, false>(hipStream_t, bf16 const *, bf16 const *, bf16 *, int, int, int, int64_t,
                                                        int64_t, int64_t, GemmEpilogue const &);
extern template hipError_t pick_bf16_tail<false, true>(hipStream_t, bf16 const *, bf16 const *, bf16 *, int, int, int, int64_t,
                                                       int64_t, int64_t, GemmEpilogue const &);
extern template hipError_t pick_bf16_group<true, false>(hipStream_t, GemmProblem const *, int, int, bool, ColreduceBatch *);

// ---------------------------------------------------------------------------
// Plain kernel for bf16 shapes the tiled kernel cannot take.
// ---------------------------------------------------------------------------
// LANES lanes an output share its reduction: a wave from 64 terms on (one thread walking 841 terms
// took 95 us for 17 x 43 outputs, its loads one behind the other; a wave 5).
template <int LANES = 64>
__global__ __launch_bounds__(256) void gemm_bf16_plain_kernel(
    bf16 const *__restrict__ A, bf16 const *__restrict__ B, bf16 *C, int M,
    int N, int K, int64_t lda, int64_t ldb, int64_t ldc, int ta, int tb,
    bf16 const *__restrict__ bias, int act, int accumulate) {
  int64_t idx = ((int64_t)blockIdx.x * 256 + threadIdx.x) / LANES;
  if (idx >= (int64_t)M * N) return;  // uniform over the LANES lanes
  int m = (int)(idx / N), n = (int)(idx % N);
  float acc = 0.0f;
  for (int k = threadIdx.x % LANES; k < K; k += LANES) {
    float a = VecIO<bf16>::load1(ta ? A + (int64_t)k * lda + m : A + (int64_t)m * lda + k);
    float b = VecIO<bf16>::load1(tb ? B + (int64_t)n * ldb + k : B + (int64_t)k * ldb + n);
    acc += a * b;
  }
#pragma unroll
  for (int off = LANES / 2; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
  if (threadIdx.x % LANES != 0) return;
  if (bias != nullptr) acc += VecIO<bf16>::load1(bias + n);
  acc = apply_activation(acc, act);
  bf16 *dst = C + (int64_t)m * ldc + n;
  if (accumulate) acc += VecIO<bf16>::load1(dst);
  VecIO<bf16>::store1(dst, acc);
}

// ---------------------------------------------------------------------------
// Column sums (bias gradient): out[n] (+)= sum_m X[m,n]
// ---------------------------------------------------------------------------
// First pass: a thread reads 16 bytes (8 bf16 / 4 fp32 columns) of kColsumRowsPerLane rows, all
// loads independent; 64 threads span the columns, the 4 row lanes of the workgroup meet in LDS.
// What is summed, and on the way written to G, is given by OP:
//   kSumOnly   X itself (nothing written)
//   kSumDrop   the dropout's backward of X, rounded as stored (dense, ldx == N: a lane's V elements
//              are a Philox block or half of one)
//   kSumAct    act'(Y) * X, rounded as stored: the gradient before a Linear's activation (for an
//              activation of "none" a copy).  ldg may be longer than a row: the columns behind it up
//              to the next whole 16 bytes become zeros, for readers that take 16 bytes at a time.
// ANY: rows of any length at any address.
// Memory bound.  [2048, 50257] bf16 at odd addresses: the copy with its sums 83 us (5 TB/s); the
// sums alone took 95 us one element at a time.
enum ColsumOp { kSumOnly = 0, kSumDrop = 1, kSumAct = 2 };
template <typename T>
struct ColsumArgs {
  T const *X, *Y;
  T *G;
  int64_t ldx, ldg;
  int M, N, rows_per_split;
  float *partials;  // nullptr: no sums wanted
  DropoutParams drop;
  int relu_mode;
};
template <typename T, int OP, int ACT, bool ANY>
__global__ __launch_bounds__(256) void colsum_partial_vec_kernel(ColsumArgs<T> a) {
  constexpr int V = VecIO<T>::kVec;
  __shared__ float red[4][64][V + 1];
  int const cx = threadIdx.x & 63;
  int const ry = threadIdx.x >> 6;
  int const n = (blockIdx.x * 64 + cx) * V;
  int const r0 = blockIdx.y * a.rows_per_split;
  int const r1 = min(a.M, r0 + a.rows_per_split);
  int const N = a.N;
  int const exist = ANY ? min(V, N - n) : V;  // of this thread's columns
  float s[V];
#pragma unroll
  for (int e = 0; e < V; e++) s[e] = 0.0f;
  auto load = [&](T const *p) -> u32x4 {
    if constexpr (ANY) return exist == V ? load_raw_any(p) : load_raw_first(p, exist);
    return load_raw_stream(p);
  };
  if (n < N) {
    for (int m0 = r0 + ry * kColsumRowsPerLane; m0 < r1; m0 += kColsumRowsPerBlock) {
      u32x4 x[kColsumRowsPerLane], y[kColsumRowsPerLane];
#pragma unroll
      for (int i = 0; i < kColsumRowsPerLane; i++) {
        int64_t const m = min(m0 + i, r1 - 1);  // clamped rows are masked below
        x[i] = load(a.X + m * a.ldx + n);
        if constexpr (OP == kSumAct && ACT != FFK_ACT_NONE) y[i] = load(a.Y + m * a.ldx + n);
      }
#pragma unroll
      for (int i = 0; i < kColsumRowsPerLane; i++) {
        if (m0 + i < r1) {
          float v[V];
          unpack_raw(x[i], v, (T const *)nullptr);
          if constexpr (OP == kSumDrop) {
            uint64_t const e0 = a.drop.offset + (uint64_t)(m0 + i) * (uint64_t)N + (uint64_t)n;
            uint32_t w[4];
            philox4x32_10(e0 >> 3, a.drop.key, w);
            if (V == 4 && (e0 & 4)) {  // upper half of the block
              w[0] = w[2];
              w[1] = w[3];
            }
#pragma unroll
            for (int e = 0; e < V; e++) v[e] = storage_round<T>(keep(w, e, a.drop) ? v[e] * a.drop.scale : 0.0f);
            VecIO<T>::store(a.G + (int64_t)(m0 + i) * a.ldg + n, v);
          }
          if constexpr (OP == kSumAct) {
            if constexpr (ACT != FFK_ACT_NONE) {
              float out[V];
              unpack_raw(y[i], out, (T const *)nullptr);
#pragma unroll
              for (int e = 0; e < V; e++) v[e] = storage_round<T>(activation_grad<ACT>(a.relu_mode, out[e], v[e]));
            }
            T *const to = a.G + (int64_t)(m0 + i) * a.ldg + n;
            u32x4 const raw = pack_raw(v, (T const *)nullptr);
            if (!ANY || n + V <= a.ldg) {
              store_raw_any(to, raw);
            } else {
              store_raw_first(to, raw, exist);
            }
          }
#pragma unroll
          for (int e = 0; e < V; e++) s[e] += v[e];
        }
      }
    }
  }
  if (a.partials == nullptr) return;  // uniform over the launch
#pragma unroll
  for (int e = 0; e < V; e++) red[ry][cx][e] = s[e];
  __syncthreads();
  if (ry == 0 && n < N) {
#pragma unroll
    for (int e = 0; e < V; e++) {
      if (ANY && e >= exist) break;
      a.partials[(int64_t)blockIdx.y * N + n + e] = (red[0][cx][e] + red[1][cx][e]) + (red[2][cx][e] + red[3][cx][e]);
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
  FFK_REQUIRE(dtype == FFK_BF16 && colsum_rows_per_split(M) == kColsumRowsPerBlock,
              "colsum_finish: partials of this shape do not come from a GEMM tail");
  FFK_HIP(colreduce_launch<bf16>(st, partials, (int)ceil_div(M, kColsumRowsPerBlock), (int)N, (int)N,
                                 static_cast<bf16 *>(out), nullptr, accumulate));
  return FFK_OK;
}

int64_t colsum_partials_elems(int64_t M, int64_t N) {
  return (int64_t)colsum_splits(M) * N;
}

// The launch of one kernel of the first pass and, where sums are wanted, of the second.
template <int OP, int ACT, bool ANY, typename T>
static int colsum_launch(hipStream_t st, ColsumArgs<T> a, T *out, bool accumulate) {
  // whole row blocks per split so that only the last split has a ragged end
  a.rows_per_split = (int)colsum_rows_per_split(a.M);
  int const used = (int)ceil_div(a.M, a.rows_per_split);
  dim3 grid((unsigned)ceil_div(a.N, 64 * VecIO<T>::kVec), (unsigned)used);
  colsum_partial_vec_kernel<T, OP, ACT, ANY><<<grid, 256, 0, st>>>(a);
  FFK_CHECK_LAUNCH();
  if (out != nullptr) FFK_HIP(colreduce_launch<T>(st, a.partials, used, a.N, a.N, out, nullptr, accumulate));
  return FFK_OK;
}

template <typename T>
static int colsum_typed(hipStream_t st, T const *X, int64_t ldx, int64_t M, int64_t N, T *out, bool accumulate,
                        float *partials) {
  ColsumArgs<T> const a = {X, nullptr, nullptr, ldx, 0, (int)M, (int)N, 0, partials, {}, 0};
  bool const vec = N % VecIO<T>::kVec == 0 && ldx % VecIO<T>::kVec == 0 && aligned16(X);
  return vec ? colsum_launch<kSumOnly, FFK_ACT_NONE, false>(st, a, out, accumulate)
             : colsum_launch<kSumOnly, FFK_ACT_NONE, true>(st, a, out, accumulate);
}

template <typename T>
static int dropout_backward_colsum_typed(hipStream_t st, T const *dy, T *dx, int64_t M, int64_t N, T *out, bool accumulate,
                                         float *partials, DropoutParams const &drop) {
  if (N % VecIO<T>::kVec != 0 || !aligned16(dy) || !aligned16(dx) || (drop.offset & 7) != 0 || M >= (1ll << 31) ||
      N >= (1ll << 31)) {
    return FFK_ERR_UNSUPPORTED;  // before any launch
  }
  ColsumArgs<T> const a = {dy, nullptr, dx, N, N, (int)M, (int)N, 0, partials, drop, 0};
  return colsum_launch<kSumDrop, FFK_ACT_NONE, false>(st, a, out, accumulate);
}

template <int ACT, typename T>
static int linear_grad_act(hipStream_t st, ColsumArgs<T> const &a, T *out, bool accumulate) {
  constexpr int V = VecIO<T>::kVec;
  bool const vec = a.N % V == 0 && a.ldg % V == 0 && aligned16(a.X) && aligned16(a.Y) && aligned16(a.G);
  return vec ? colsum_launch<kSumAct, ACT, false>(st, a, out, accumulate) : colsum_launch<kSumAct, ACT, true>(st, a, out, accumulate);
}
template <typename T>
static int linear_grad_typed(hipStream_t st, int act, int relu_mode, T const *y, T const *dy, T *g, int64_t ldg, int64_t M,
                             int64_t N, T *colsum, bool accumulate, float *partials) {
  ColsumArgs<T> const a = {dy, y, g, N, ldg, (int)M, (int)N, 0, colsum != nullptr ? partials : nullptr, {}, relu_mode};
  switch (act) {
    case FFK_ACT_NONE: return linear_grad_act<FFK_ACT_NONE>(st, a, colsum, accumulate);
    case FFK_ACT_RELU: return linear_grad_act<FFK_ACT_RELU>(st, a, colsum, accumulate);
    case FFK_ACT_SIGMOID: return linear_grad_act<FFK_ACT_SIGMOID>(st, a, colsum, accumulate);
    default: return linear_grad_act<FFK_ACT_TANH>(st, a, colsum, accumulate);
  }
}

int linear_grad(hipStream_t st, int dtype, int act, int relu_mode, void const *y, void const *dy, void *g, int64_t ldg,
                int64_t M, int64_t N, void *colsum, bool accumulate, float *partials) {
  FFK_REQUIRE(M < (1ll << 31) && N < (1ll << 31), "linear_grad: dimension exceeds 2^31");
  if (dtype == FFK_FLOAT) {
    return linear_grad_typed(st, act, relu_mode, static_cast<float const *>(y), static_cast<float const *>(dy),
                             static_cast<float *>(g), ldg, M, N, static_cast<float *>(colsum), accumulate, partials);
  }
  return linear_grad_typed(st, act, relu_mode, static_cast<bf16 const *>(y), static_cast<bf16 const *>(dy),
                           static_cast<bf16 *>(g), ldg, M, N, static_cast<bf16 *>(colsum), accumulate, partials);
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
    return dropout_backward_colsum_typed(st, static_cast<float const *>(dy), static_cast<float *>(dx), M, N,
                                         static_cast<float *>(colsum), accumulate, partials, drop);
  }
  if (dtype == FFK_BF16) {
    return dropout_backward_colsum_typed(st, static_cast<bf16 const *>(dy), static_cast<bf16 *>(dx), M, N,
                                         static_cast<bf16 *>(colsum), accumulate, partials, drop);
  }
  return FFK_ERR_UNSUPPORTED;
}

// Whether a weight gradient joins a group: one that fills the chip twice over has better kernels of
// its own, and the group's take operands readable 16 bytes at a time.
static bool joins_group(int dtype, int64_t M, int64_t N, int64_t K, GemmProblem const &p, GemmEpilogue const &ep) {
  if (dtype != FFK_BF16 || gemm_variant_override() != 0 || ep.bias != nullptr || ep.activation != FFK_ACT_NONE ||
      ep.tail != GemmEpilogue::kTailNone) {
    return false;
  }
  if (M <= 0 || N <= 0 || K <= 0 || M >= (1ll << 31) || N >= (1ll << 31) || K >= (1ll << 31)) return false;
  if (!p.A || !p.B || !p.C || p.lda < M || p.ldb < N || p.ldc < N) return false;
  if (ceil_div(M, 128) * ceil_div(N, 128) >= 2 * kNumCU) return false;
  return M % 8 == 0 && N % 8 == 0 && p.lda % 8 == 0 && p.ldb % 8 == 0 && aligned16(p.A) && aligned16(p.B) &&
         edge_operands_ok(p.lda, p.ldb);
}

int weight_grad_dispatch(hipStream_t st, int dtype, int64_t M, int64_t N, int64_t K, void const *A, int64_t lda,
                         void const *B, int64_t ldb, void *C, int64_t ldc, GemmEpilogue const &ep) {
  WeightGradGroup *const g = tl_weight_grads;
  GemmProblem const p = {M, N, A, lda, B, ldb, C, ldc};
  if (g != nullptr && g->count < kMaxGemmGroup && (g->count == 0 || (g->K == K && g->accumulate == ep.accumulate)) &&
      joins_group(dtype, M, N, K, p, ep)) {
    bool clash = false;  // two gradients into one tensor keep their order
    for (int i = 0; i < g->count; i++) clash = clash || g->p[i].C == C;
    if (!clash) {
      g->p[g->count++] = p;
      g->K = K;
      g->accumulate = ep.accumulate;
      return FFK_OK;
    }
    int const rc = weight_grad_flush(st, *g);
    if (rc != FFK_OK) return rc;
  }
  return gemm_dispatch(st, dtype, true, false, M, N, K, A, lda, B, ldb, C, ldc, ep);
}

int weight_grad_flush(hipStream_t st, WeightGradGroup &g, ColreduceBatch *sums) {
  int const n = g.count;
  g.count = 0;
  if (n == 0) return FFK_OK;
  if (n == 1) {
    GemmProblem const &p = g.p[0];
    GemmEpilogue ep;
    ep.accumulate = g.accumulate;
    return gemm_dispatch(st, FFK_BF16, true, false, p.M, p.N, g.K, p.A, p.lda, p.B, p.ldb, p.C, p.ldc, ep);
  }
  hipError_t const e = pick_bf16_group<true, false>(st, g.p, n, (int)g.K, g.accumulate, sums);
  FFK_HIP(e);
  return FFK_OK;
}

bool gemm_tail_supported(int dtype, bool ta, bool tb, int64_t M, int64_t N, int64_t K,
                         void const *A, int64_t lda, void const *B, int64_t ldb,
                         void const *C, int64_t ldc, GemmEpilogue const &ep) {
  if (dtype != FFK_BF16 || ta || ep.accumulate || ldc != N || M <= 0 || N <= 0 || K <= 0) return false;
  if (M >= (1ll << 31) || N >= (1ll << 31) || K >= (1ll << 31)) return false;
  if ((ep.tail_dropout.offset & 7) != 0) return false;
  bool sums = false;
  switch (ep.tail) {
    case GemmEpilogue::kTailGeluDropout:
    case GemmEpilogue::kTailActDropout:
      if (!tb || ep.tail_out == nullptr || !aligned16(ep.tail_out)) return false;
      break;
    case GemmEpilogue::kTailDropoutGeluGrad:
    case GemmEpilogue::kTailDropoutReluGrad:
      if (tb || ep.tail_in == nullptr || !aligned16(ep.tail_in)) return false;
      sums = true;
      if (ep.tail_colsum_partials != nullptr && colsum_rows_per_split(M) != kColsumRowsPerBlock) return false;
      break;
    case GemmEpilogue::kTailDropoutAdd:
      if (ep.tail_in == nullptr || !aligned16(ep.tail_in) || (!tb && !ep.tail_any_size)) return false;
      break;
    default: return false;
  }
  int const variant = gemm_variant_override();
  bool const vec_ok = (K % 8 == 0) && (lda % 8 == 0) && (ldb % 8 == 0) && aligned16(A) && aligned16(B) &&
                      (tb || N % 8 == 0);
  if (!vec_ok) return false;
  if (pipe_tile_for(static_cast<bf16 const *>(C), (int)M, (int)N, (int)K, lda, ldb, ldc, ep, variant) != 0) {
    // with one 256x256 or 128x128 tile a CU every CU reaches its store at the same time and nothing
    // overlaps GELU's arithmetic: two kernels are as soon done
    return !(ep.tail_any_size && ep.tail == GemmEpilogue::kTailGeluDropout);
  }
  if (!ep.tail_any_size || variant != 0 || N % 8 != 0 || !aligned16(C) || !edge_operands_ok(lda, ldb)) return false;
  bool const splits = gemm_split_tile((int)M, (int)N, (int)K, ep) != 0;
  if (ep.tail == GemmEpilogue::kTailGeluDropout) return splits;
  return splits || sums || (M >= 128 && N >= 128);
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
    e = gemm_f32_launch(st, ta, tb, (int)M, (int)N, (int)K, static_cast<float const *>(A), lda,
                        static_cast<float const *>(B), ldb, static_cast<float *>(C), ldc, ep);
  } else if (dtype == FFK_BF16) {
    FFK_REQUIRE(ep.tail == GemmEpilogue::kTailNone ||
                    gemm_tail_supported(dtype, ta, tb, M, N, K, A, lda, B, ldb, C, ldc, ep),
                "gemm: this shape has no fused tail (ask gemm_tail_supported first)");
    bf16 const *a = static_cast<bf16 const *>(A);
    bf16 const *b = static_cast<bf16 const *>(B);
    bf16 *c = static_cast<bf16 *>(C);
    // 16-byte chunks: the contiguous extent of each operand (K, or M / N) must be a multiple of 8
    // elements, or padded to one, rows 16-byte aligned.
    bool vec_ok = ((ta ? M % 8 == 0 : K % 8 == 0) || (ep.a_padded && !tb)) && (tb ? K % 8 == 0 : N % 8 == 0) && (lda % 8 == 0) &&
                  (ldb % 8 == 0) && aligned16(A) && aligned16(B) && K > 0;
    // Operands that are not: the register-staged kernel, but for products of so few elements that
    // one thread, or one wave, an output is over as soon.
    // (A reduction of thousands over a few 64 x 64 tiles would be walked by as many workgroups: 52 x 37 over
    // 1907 51 us so, 13 with a wave an output.)
    bool const few = K >= 512 && M * N <= 4 * 64 * 64 && M * N * K < (1 << 23);
    if (!vec_ok && (K == 0 || M * N * K < (1 << 21) || (few && ep.tail == GemmEpilogue::kTailNone))) {
      int64_t const total = M * N * (K >= 64 ? 64 : 1);
      if (describe_only(K >= 64 ? "gemm_bf16_plain_kernel" : "gemm_bf16_plain_kernel<1>")) return FFK_OK;
      auto kern = K >= 64 ? gemm_bf16_plain_kernel<64> : gemm_bf16_plain_kernel<1>;
      kern<<<(unsigned)ceil_div(total, 256), 256, 0, st>>>(
          a, b, c, (int)M, (int)N, (int)K, lda, ldb, ldc, ta, tb,
          static_cast<bf16 const *>(ep.bias), ep.activation, ep.accumulate);
      e = hipGetLastError();
    } else if (ep.tail != GemmEpilogue::kTailNone) {
      e = tb ? pick_bf16_tail<false, true>(st, a, b, c, (int)M, (int)N, (int)K, lda, ldb, ldc, ep)
             : pick_bf16_tail<false, false>(st, a, b, c, (int)M, (int)N, (int)K, lda, ldb, ldc, ep);
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
