// bf16 GEMM kernels for C = A^T . B (weight gradients).
#include "gemm_bf16.h"

namespace ffk {
template hipError_t pick_bf16<true, false>(hipStream_t, bf16 const *, bf16 const *, bf16 *, int, int, int, int64_t, int64_t,
                                      int64_t, GemmEpilogue const &, bool);
template hipError_t pick_bf16_group<true, false>(hipStream_t, GemmProblem const *, int, int, bool, ColreduceBatch *);
}  // namespace ffk
