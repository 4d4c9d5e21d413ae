// The backward of a bf16 Linear layer in one launch, or two: tiles of the input gradient and of the
// weight gradient as jobs of one grid, the activation's gradient applied to the output gradient on its
// way into LDS, and the bias gradient summed by the tiles of the weight gradient's first column from the
// pieces they stage anyway.  No gradient copy, no column-sum launches.  The second launch is there where
// a reduction is split over workgroups: it adds up the partial sums of all three gradients.
// Small layers are bound by the launches, four or five before (64 x 128 -> 40 17 us with the forward, 9 now),
// long reductions over few outputs by the few workgroups that walked them (5533 x 116 -> 134: the weight
// gradient's 87 k-tiles on six, 213 us; 21 now).
#include "linear_any.h"
#include "gemm_any.h"
#include <algorithm>

namespace ffk {

namespace {

struct LinearAnyJobs {
  LinearAnyArgs a;
  int blocks_dx;  // workgroups of the input gradient
  int per_dx, per_dw;
  float *part_dx, *part_dw, *part_db;  // [split][elements], nullptr: the reduction is not split
};

// 64x64 tiles on four waves, of which three workgroups share a CU (while one waits at a barrier or for its
// loads the others multiply), or 128x128 tiles on eight, two workgroups a CU.
template <int ACT, int T>
__global__ __launch_bounds__(T * 4) void linear_any_bwd_kernel(LinearAnyJobs p) {
  using DxTile = AnyTile<T, T, T / 2, 32, true, false, ACT>;
  using DwTile = AnyTile<T, T, T / 2, 32, false, false, ACT>;
  constexpr int kElems = DxTile::kBufElems > DwTile::kBufElems ? DxTile::kBufElems : DwTile::kBufElems;
  __shared__ __attribute__((aligned(16))) bf16 smem[2 * kElems];
  int const I = p.a.in_dim, O = p.a.out_dim, B = p.a.batch, t = threadIdx.x;
  int const nbn = (I + T - 1) / T;
  auto add_to = [](bf16 *dst, float v, bool accumulate) __attribute__((always_inline)) {
    VecIO<bf16>::store1(dst, accumulate ? v + VecIO<bf16>::load1(dst) : v);
  };
  if ((int)blockIdx.x < p.blocks_dx) {
    // input_grad[batch, in] (+)= g[batch, out] . weight[out, in]
    int const tiles = ((B + T - 1) / T) * nbn, split = blockIdx.x / tiles, tile = blockIdx.x - split * tiles;
    int const m0 = tile / nbn * T, n0 = tile % nbn * T, KT = (O + kBK - 1) / kBK, kt0 = split * p.per_dx;
    typename DxTile::OpA a;
    typename DxTile::OpB b;
    a.init(p.a.dy, p.a.y, O, B, O, p.a.relu_mode, m0, t);
    b.init(p.a.w, nullptr, I, I, O, 0, n0, t);
    DxTile x;
    x.template reduce<false>(a, b, O, kt0, min(kt0 + p.per_dx, KT), smem);
    if (p.part_dx != nullptr) {
      float *const to = p.part_dx + (int64_t)split * B * I;
      x.store(m0, n0, B, I, [&](int m, int n, float v) { to[(int64_t)m * I + n] = v; });
    } else {
      bool const acc = (p.a.accumulate & FFK_ACC_INPUT) != 0;
      x.store(m0, n0, B, I, [&](int m, int n, float v) { add_to(p.a.dx + (int64_t)m * I + n, v, acc); });
    }
  } else {
    // weight_grad[out, in] (+)= g[batch, out]^T . input[batch, in]; bias_grad[out] (+)= column sums of g
    int const bid = blockIdx.x - p.blocks_dx;
    int const nbw = p.a.dw != nullptr ? nbn : 1;  // (column sums alone: one column of tiles)
    int const tiles = ((O + T - 1) / T) * nbw, split = bid / tiles, tile = bid - split * tiles;
    int const m0 = tile / nbw * T, n0 = tile % nbw * T, KT = (B + kBK - 1) / kBK, kt0 = split * p.per_dw;
    int const kt1 = min(kt0 + p.per_dw, KT);
    typename DwTile::OpA a;
    typename DwTile::OpB b;
    a.init(p.a.dy, p.a.y, O, O, B, p.a.relu_mode, m0, t);
    b.init(p.a.x, nullptr, I, I, B, 0, n0, t);
    DwTile x;
    bool const sums = p.a.db != nullptr && n0 == 0;  // uniform over the workgroup
    if (sums) {
      x.template reduce<true>(a, b, B, kt0, kt1, smem);
    } else {
      x.template reduce<false>(a, b, B, kt0, kt1, smem);
    }
    if (p.a.dw != nullptr) {
      if (p.part_dw != nullptr) {
        float *const to = p.part_dw + (int64_t)split * O * I;
        x.store(m0, n0, O, I, [&](int m, int n, float v) { to[(int64_t)m * I + n] = v; });
      } else {
        bool const acc = (p.a.accumulate & FFK_ACC_WEIGHT) != 0;
        x.store(m0, n0, O, I, [&](int m, int n, float v) { add_to(p.a.dw + (int64_t)m * I + n, v, acc); });
      }
    }
    if (sums) {
      bool const acc = (p.a.accumulate & FFK_ACC_BIAS) != 0;
      x.store_sums(m0, O, smem, [&](int m, float v) {
        if (p.part_db != nullptr) {
          p.part_db[(int64_t)split * O + m] = v;
        } else {
          add_to(p.a.db + m, v, acc);
        }
      });
    }
  }
}

struct LinearAnyFinish {
  struct Sum {
    float const *part;
    bf16 *out;
    int64_t elems;
    int splits, accumulate;
  } s[3];
  int64_t first[3];  // workgroup of the first element of each
};

// An element a thread; 256 elements of one gradient a workgroup.
__global__ __launch_bounds__(256) void linear_any_finish_kernel(LinearAnyFinish f) {
  int const q = (int64_t)blockIdx.x >= f.first[2] ? 2 : (int64_t)blockIdx.x >= f.first[1] ? 1 : 0;
  float const *part = f.s[q].part;
  int64_t const elems = f.s[q].elems, i = ((int64_t)blockIdx.x - f.first[q]) * 256 + threadIdx.x;
  int const splits = f.s[q].splits;
  if (i >= elems) return;
  float sum = 0.0f;
  for (int k = 0; k < splits; k += 8) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; u++) v[u] = k + u < splits ? part[(k + u) * elems + i] : 0.0f;
#pragma unroll
    for (int u = 0; u < 8; u++) sum += v[u];
  }
  bf16 *const dst = f.s[q].out + i;
  VecIO<bf16>::store1(dst, f.s[q].accumulate ? sum + VecIO<bf16>::load1(dst) : sum);
}

}  // namespace

// 64x64 or 128x128.  The large tiles read LDS half as often for a multiplication, but want four times the
// work to fill the chip, and columns to fill (2048 x 206 -> 34294 660 us on the small ones, 488 on the large).
static int any_tile_for(int64_t batch, int64_t in_dim, int64_t out_dim) {
  int64_t const k_tiles = ceil_div(batch, 64) * ceil_div(in_dim, 64) * ceil_div(out_dim, 64);
  return in_dim > 64 && k_tiles > 8000 ? 128 : 64;
}

LinearAnyPlan linear_any_plan(int64_t batch, int64_t in_dim, int64_t out_dim, size_t max_scratch) {
  LinearAnyPlan p;
  p.tile = any_tile_for(batch, in_dim, out_dim);
  int64_t const nbn = ceil_div(in_dim, p.tile), tx = ceil_div(batch, p.tile) * nbn, tw = ceil_div(out_dim, p.tile) * nbn;
  int64_t const kx = ceil_div(out_dim, kBK), kw = ceil_div(batch, kBK);
  // Even shares of the k-tiles for two and a half workgroups a CU (two of the large).
  int64_t const share = std::max(kLinearAnyShare, ceil_div(tx * kx + tw * kw, p.tile == 64 ? kNumCU * 5 / 2 : kNumCU * 2));
  auto cut = [&](int64_t k, int &splits, int &per) {
    int64_t const s = k * 2 <= share * 3 ? 1 : ceil_div(k, share);
    per = (int)ceil_div(k, s);
    splits = (int)ceil_div(k, per);
  };
  cut(kx, p.splits_dx, p.per_dx);
  cut(kw, p.splits_dw, p.per_dw);
  auto bytes = [&] {
    return (size_t)4 * ((p.splits_dx > 1 ? (size_t)p.splits_dx * batch * in_dim : 0) +
                        (p.splits_dw > 1 ? (size_t)p.splits_dw * out_dim * (in_dim + 1) : 0));
  };
  while ((p.scratch = bytes()) > max_scratch) {
    // fewer parts of whichever sums take more room
    bool const dx = (int64_t)p.splits_dx * batch >= (int64_t)p.splits_dw * out_dim;
    int &s = (dx && p.splits_dx > 1) || p.splits_dw == 1 ? p.splits_dx : p.splits_dw;
    int64_t const k = &s == &p.splits_dx ? kx : kw;
    int &per = &s == &p.splits_dx ? p.per_dx : p.per_dw;
    per = (int)ceil_div(k, s - 1);
    s = (int)ceil_div(k, per);
  }
  return p;
}

template <int T>
static void launch_jobs(hipStream_t st, int activation, unsigned blocks, LinearAnyJobs const &j) {
  switch (activation) {
    case FFK_ACT_RELU: linear_any_bwd_kernel<FFK_ACT_RELU, T><<<blocks, T * 4, 0, st>>>(j); break;
    case FFK_ACT_SIGMOID: linear_any_bwd_kernel<FFK_ACT_SIGMOID, T><<<blocks, T * 4, 0, st>>>(j); break;
    case FFK_ACT_TANH: linear_any_bwd_kernel<FFK_ACT_TANH, T><<<blocks, T * 4, 0, st>>>(j); break;
    default: linear_any_bwd_kernel<FFK_ACT_NONE, T><<<blocks, T * 4, 0, st>>>(j); break;
  }
}

hipError_t linear_any_backward(hipStream_t st, int activation, LinearAnyArgs const &a, LinearAnyPlan const &plan, void *scratch) {
  LinearAnyJobs j = {};
  j.a = a;
  int64_t const nbn = ceil_div(a.in_dim, plan.tile);
  j.per_dx = plan.per_dx;
  j.per_dw = plan.per_dw;
  j.blocks_dx = a.dx != nullptr ? (int)(ceil_div(a.batch, plan.tile) * nbn * plan.splits_dx) : 0;
  int const blocks_dw = (int)(ceil_div(a.out_dim, plan.tile) * (a.dw != nullptr ? nbn : a.db != nullptr ? 1 : 0) * plan.splits_dw);
  float *at = static_cast<float *>(scratch);
  if (plan.splits_dx > 1) {
    j.part_dx = at;
    at += (int64_t)plan.splits_dx * a.batch * a.in_dim;
  }
  if (plan.splits_dw > 1) {
    j.part_dw = at;
    j.part_db = at + (int64_t)plan.splits_dw * a.out_dim * a.in_dim;
  }
  unsigned const blocks = (unsigned)(j.blocks_dx + blocks_dw);
  if (plan.tile == 64) {
    launch_jobs<64>(st, activation, blocks, j);
  } else {
    launch_jobs<128>(st, activation, blocks, j);
  }
  hipError_t const e = hipGetLastError();
  if (e != hipSuccess) return e;
  LinearAnyFinish f = {};
  int64_t groups = 0;
  auto add = [&](int q, bool wanted, float const *part, bf16 *out, int64_t elems, int splits, int acc) {
    f.first[q] = groups;
    if (!wanted) return;
    f.s[q] = {part, out, elems, splits, (a.accumulate & acc) != 0};
    groups += ceil_div(elems, 256);
  };
  add(0, plan.splits_dx > 1 && a.dx != nullptr, j.part_dx, a.dx, (int64_t)a.batch * a.in_dim, plan.splits_dx, FFK_ACC_INPUT);
  add(1, plan.splits_dw > 1 && a.dw != nullptr, j.part_dw, a.dw, (int64_t)a.out_dim * a.in_dim, plan.splits_dw, FFK_ACC_WEIGHT);
  add(2, plan.splits_dw > 1 && a.db != nullptr, j.part_db, a.db, a.out_dim, plan.splits_dw, FFK_ACC_BIAS);
  if (groups == 0) return hipSuccess;
  linear_any_finish_kernel<<<(unsigned)groups, 256, 0, st>>>(f);
  return hipGetLastError();
}

}  // namespace ffk
