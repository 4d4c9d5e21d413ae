// The backward of a bf16 Linear layer on the tiles of gemm_any.h (linear_any.hip).
#pragma once
#include "ffk_common.h"
#include <algorithm>

namespace ffk {

struct LinearAnyPlan {
  int tile;                                  // 64 or 128, square
  int splits_dx, per_dx, splits_dw, per_dw;  // parts of each reduction, 64-deep k-tiles of a part
  size_t scratch;                            // bytes of partial sums
};
// The fewest k-tiles of a part, 5 us: the second launch takes about 4.  A reduction of up to half as many again stays whole.
constexpr int64_t kLinearAnyShare = 12;
inline bool linear_any_may_split(int64_t batch, int64_t out_dim) {
  return ceil_div(std::max(batch, out_dim), 64) * 2 > kLinearAnyShare * 3;
}
// How the two reductions (over out_dim and over batch) are cut; with no more than max_scratch bytes.
LinearAnyPlan linear_any_plan(int64_t batch, int64_t in_dim, int64_t out_dim, size_t max_scratch);

struct LinearAnyArgs {
  bf16 const *y, *dy, *x, *w;
  bf16 *dx, *dw, *db;  // nullptr: not wanted
  int batch, in_dim, out_dim, relu_mode, accumulate;
};
hipError_t linear_any_backward(hipStream_t stream, int activation, LinearAnyArgs const &args, LinearAnyPlan const &plan,
                               void *scratch);

}  // namespace ffk
