// bf16 GEMM kernels for C = A . B^T (forward) with element-wise operators on the tile store.
#include "gemm_bf16.h"

namespace ffk {
template hipError_t pick_bf16_tail<false, true>(hipStream_t, bf16 const *, bf16 const *, bf16 *, int, int, int, int64_t, int64_t,
                                           int64_t, GemmEpilogue const &);
}  // namespace ffk
