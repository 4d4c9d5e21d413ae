// Internal GEMM interface shared by Linear, the attention projections and the
// public ffk_gemm entry point.
#pragma once
#include "ffk_common.h"
#include "dropout_rng.h"

namespace ffk {

// The gradient before a Linear's activation, from its output y and output gradient dy.
template <int ACT>
__device__ __forceinline__ float activation_grad(int relu_mode, float y, float dy) {
  if (ACT == FFK_ACT_NONE) return dy;
  if (ACT == FFK_ACT_RELU) {
    if (relu_mode == 1) return dy > 0.0f ? 1.0f : 0.0f;  // linear_kernels_cpu.cc:46-52,69-71
    return y > 0.0f ? dy : 0.0f;                         // cuda_helper.cu:60-64
  }
  if (ACT == FFK_ACT_SIGMOID) return dy * y * (1.0f - y);  // cuda_helper.cu:87-91
  return dy * (1.0f - y * y);                              // tanh
}

struct GemmEpilogue {
  void const *bias = nullptr;  // [N] in the GEMM dtype, added to every row
  int activation = FFK_ACT_NONE;
  bool accumulate = false;     // C += result instead of C = result
  // A's rows (M or K elements) are followed by zeros up to the next multiple of 8 elements, which
  // belong to its memory (bf16, trans_b == false): it is read 16 bytes at a time whatever the length
  bool a_padded = false;
  // Optional scratch for split-K, used when the output has too few tiles to occupy the chip: as many
  // splits as it has room for fp32 copies of the output, and as help.
  void *splitk_ws = nullptr;
  size_t splitk_ws_bytes = 0;
  // Optional element-wise operators applied to the output tile while it is
  // written (bf16 only, see gemm_tail_supported).  With a tail the GEMM gives
  // the bits of the separate kernels run after it:
  //   kTailGeluDropout     C = result (kept: backward reads the pre-activation),
  //                        tail_out = dropout(GELU(C))
  //   kTailDropoutGeluGrad C = dropout_backward(result) * GELU'(tail_in); the
  //                        plain result is not stored
  //   kTailDropoutAdd      C = tail_in + dropout(result); the plain result is
  //                        not stored
  //   kTailDropoutReluGrad C = dropout_backward(result) where tail_in > 0, else 0
  //   kTailActDropout      C = act(result), tail_out = dropout(C)
  // tail_in / tail_out are dense [M, N] tensors, the dropout stream is indexed
  // by m * N + n from tail_dropout.offset.
  enum Tail { kTailNone = 0, kTailGeluDropout = 1, kTailDropoutGeluGrad = 2, kTailDropoutAdd = 3,
              kTailDropoutReluGrad = 4, kTailActDropout = 5 };
  int tail = kTailNone;
  // also sizes that are no whole tiles, or fewer than fill the chip (the encoder layer; the entry
  // points keep to the sizes they document)
  bool tail_any_size = false;
  void const *tail_in = nullptr;
  void *tail_out = nullptr;
  DropoutParams tail_dropout = {};
  // kTailDropout*Grad, optional: the GEMM also leaves the partial column
  // sums of what it stores (colsum_partials_elems(M, N) floats, the partials
  // colsum_dispatch would compute from the stored tensor); colsum_finish adds
  // them up into the column sums (+)= out.
  float *tail_colsum_partials = nullptr;
};
int colsum_finish(hipStream_t stream, int dtype, float const *partials, int64_t M, int64_t N, void *out,
                  bool accumulate);

// Whether gemm_dispatch can run this GEMM with ep.tail (it fails otherwise).
bool gemm_tail_supported(int dtype, bool trans_a, bool trans_b, int64_t M, int64_t N,
                         int64_t K, void const *A, int64_t lda, void const *B, int64_t ldb,
                         void const *C, int64_t ldc, GemmEpilogue const &ep);

// C[M,N] (+)= op(A) . op(B), fp32 accumulation.
//   trans_a == false: A is [M,K] row-major (lda = K); true: A is [K,M] (lda = M)
//   trans_b == false: B is [K,N] row-major (ldb = N); true: B is [N,K] (ldb = K)
// lda/ldb/ldc are row strides in elements (>= the dense value), so strided
// views (column slices of a fused buffer) can be used directly.
int gemm_dispatch(hipStream_t stream, int dtype, bool trans_a, bool trans_b,
                  int64_t M, int64_t N, int64_t K, void const *A, int64_t lda,
                  void const *B, int64_t ldb, void *C, int64_t ldc,
                  GemmEpilogue const &ep);

// Weight gradients that are collected and run as ONE launch: C = A^T . B, A [K, M], B [K, N], of
// problems with the same reduction length K that each leave part of the chip idle.  While a group
// is set on the calling thread, weight_grad_dispatch puts such problems into it instead of launching
// them (their operands have to stay as they are until the flush), and launches all others as
// gemm_dispatch would.
constexpr int kMaxGemmGroup = 4;
struct GemmProblem {
  int64_t M, N;
  void const *A;
  int64_t lda;
  void const *B;
  int64_t ldb;
  void *C;
  int64_t ldc;
};
struct WeightGradGroup {
  GemmProblem p[kMaxGemmGroup];
  int count = 0;
  int64_t K = 0;
  bool accumulate = false;
};
inline thread_local WeightGradGroup *tl_weight_grads = nullptr;
// Collects the calling thread's weight gradients for its lifetime (unless an outer one does).
struct CollectWeightGrads {
  WeightGradGroup group;
  WeightGradGroup *const saved;
  explicit CollectWeightGrads(bool on) : saved(tl_weight_grads) {
    if (on && saved == nullptr) tl_weight_grads = &group;
  }
  ~CollectWeightGrads() { tl_weight_grads = saved; }
};
// Set while an encoder layer's entry point runs its operators on the calling thread: its Linear backwards then run as
// a sequence of products, whose bits the fused operators and the sequence of single ones share, and not as the jobs of
// one launch (linear_any.hip), which add up in another order.
inline thread_local bool tl_layer_operators = false;
struct LayerOperators {
  bool const saved = tl_layer_operators;
  LayerOperators() { tl_layer_operators = true; }
  ~LayerOperators() { tl_layer_operators = saved; }
};
int weight_grad_dispatch(hipStream_t stream, int dtype, int64_t M, int64_t N, int64_t K, void const *A, int64_t lda,
                         void const *B, int64_t ldb, void *C, int64_t ldc, GemmEpilogue const &ep);
// Runs what was collected (nothing to do for an empty group) and empties it.  sums: column reductions, complete
// but for this pass, that may run in the same launch; it empties what it has taken.
struct ColreduceBatch;
int weight_grad_flush(hipStream_t stream, WeightGradGroup &group, ColreduceBatch *sums = nullptr);

// out[N] (+)= sum over the M rows of X[M,N] (ldx row stride); `partials` is
// fp32 scratch of colsum_partials_elems(M, N) floats.
int64_t colsum_partials_elems(int64_t M, int64_t N);
// dx[M,N] = dropout_backward(dy) and colsum (+)= its column sums (the bias
// gradient of the Linear whose output the dropout follows), one pass over dy.
// The sums are taken over dx as stored, in the order colsum_dispatch uses, so
// they are the bits of the two separate kernels.  FFK_ERR_UNSUPPORTED (nothing
// launched, no message) when the shape has no vector kernel.
int dropout_backward_colsum(hipStream_t stream, int dtype, void const *dy, void *dx, int64_t M,
                            int64_t N, void *colsum, bool accumulate, float *partials,
                            DropoutParams const &drop);
// g[M,N] = act'(y) * dy (activation none: a copy) with rows of ldg elements, and colsum (+)= the column
// sums of what is stored (nullptr: not wanted), one pass over dy and y; the columns of g from N to the
// next whole 16 bytes, if ldg has them, become zeros.
int linear_grad(hipStream_t stream, int dtype, int activation, int relu_mode, void const *y, void const *dy, void *g,
                int64_t ldg, int64_t M, int64_t N, void *colsum, bool accumulate, float *partials);
int colsum_dispatch(hipStream_t stream, int dtype, void const *X, int64_t ldx,
                    int64_t M, int64_t N, void *out, bool accumulate,
                    float *partials);

}  // namespace ffk
