// Linear forward/backward for gfx950.
//
// forward : output = act(input . weight^T + bias), bias and activation fused
//           into the GEMM epilogue (the reference runs a second rank-1 GEMM for
//           the bias, lib/kernels/src/cuda/ops/linear_kernels.cu:163, and never
//           applies the activation on the GPU, :183-200; its CPU path does,
//           lib/kernels/src/kernels/linear_kernels_cpu.cc:33-42).
// backward: g = act'(.) * output_grad into the caller's workspace (the
//           reference cudaMallocs a copy of output_grad per call,
//           lib/kernels/src/kernels/linear_kernels.cc:104-106), then three
//           products: input_grad (+)= g . W, weight_grad (+)= g^T . X,
//           bias_grad (+)= column sums of g (linear_kernels.cu:249-334).
#include "elementwise.h"
#include "gemm.h"
#include "fused_ops.h"
#include "small_f32.h"
#include "colreduce.h"
#include "linear_any.h"

namespace ffk {

static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// in = (weight, weight_grad); out = weight_grad + lambda * weight
struct L2RegGrad {
  float lambda;
  __device__ __forceinline__ void operator()(float const (&in)[2], float (&out)[1]) const {
    out[0] = in[1] + lambda * in[0];
  }
};

template <typename T>
static hipError_t l2_reg_grad(hipStream_t st, void const *w, void *dw, int64_t n, float lambda) {
  EwArgs<T, 2, 1> a;
  a.in[0] = static_cast<T const *>(w);
  a.in[1] = static_cast<T const *>(dw);
  a.in_elems[0] = n;
  a.in_elems[1] = n;
  a.out[0] = static_cast<T *>(dw);
  a.n = n;
  return ew_launch<T, 2, 1>(st, a, L2RegGrad{lambda});
}

// ---------------------------------------------------------------------------
// Small fp32 Linear layers: ONE launch forward and ONE backward on the tiles of small_f32.h.  At
// sizes like the reference's CPU-runnable case ([32,64] . [128,64]^T) a pass is one chain of
// latencies around almost no work: 6.5 + 7.2 us with 64x64 tiles staged through LDS and one wave's
// chain of 32 MFMAs, 2.4 + 2.9 us with these.
// The backward's jobs -- tiles of input_grad, then tiles of weight_grad, the first column of which
// also adds up bias_grad -- are independent given (output, output_grad): g = act'(output) *
// output_grad is applied where an operand element is used, never stored.
// ---------------------------------------------------------------------------
struct SmallLinearBwd {
  float const *y, *dy, *x, *w;
  float *dx, *dw, *db;
  int batch, in_dim, out_dim;
  int relu_mode, accumulate;  // accumulate: FFK_ACC_* bits
  int blocks_dx;
};
struct SmallLinearFwd {
  float const *x, *w, *bias;
  float *y;
  int batch, in_dim, out_dim, act;
};

// WAVES waves a workgroup; a tile of input_grad (reduction out_dim) takes SX of them, a tile of
// weight_grad (reduction batch) all: a long batch over a small weight needs many waves a tile.
template <int T, int ACT, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void linear_small_bwd_f32_kernel(SmallLinearBwd p) {
  __shared__ SmallShared<T, WAVES> sm;
  constexpr int SX = 4;
  int const bid = blockIdx.x;
  int const nbn = (p.in_dim + T - 1) / T;
  auto no_bias = [](int, float) {};
  if (bid < p.blocks_dx) {
    // input_grad[batch, in] (+)= g[batch, out] . weight[out, in]
    int const tile = bid * (WAVES / SX) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) / SX;
    int const tm = tile / nbn;
    SmallOperand<true, ACT> const a = {p.dy, p.y, p.out_dim, p.relu_mode};
    SmallOperand<false, FFK_ACT_NONE> const b = {p.w, nullptr, p.in_dim, 0};
    auto store = [&](int m, int n, float v) { p.dx[(int64_t)m * p.in_dim + n] = v; };
    small_tile<T, SX, WAVES>(a, b, p.batch, p.in_dim, p.out_dim, tm * T, (tile - tm * nbn) * T, tm * T < p.batch,
                             (p.accumulate & FFK_ACC_INPUT) != 0 ? p.dx : nullptr, p.in_dim, store, false, no_bias, sm);
  } else {
    // weight_grad[out, in] (+)= g[batch, out]^T . input[batch, in]; bias_grad[out] (+)= column sums of g
    int const tb = bid - p.blocks_dx;
    SmallOperand<false, ACT> const a = {p.dy, p.y, p.out_dim, p.relu_mode};
    SmallOperand<false, FFK_ACT_NONE> const b = {p.x, nullptr, p.in_dim, 0};
    auto store = [&](int m, int n, float v) { p.dw[(int64_t)m * p.in_dim + n] = v; };
    auto store_bias = [&](int m, float v) { p.db[m] = (p.accumulate & FFK_ACC_BIAS) != 0 ? p.db[m] + v : v; };
    small_tile<T, WAVES, WAVES>(a, b, p.out_dim, p.in_dim, p.batch, (tb / nbn) * T, (tb % nbn) * T, true,
                                (p.accumulate & FFK_ACC_WEIGHT) != 0 ? p.dw : nullptr, p.in_dim, store,
                                p.db != nullptr && tb % nbn == 0, store_bias, sm);
  }
}

// output = act(input . weight^T + bias)
template <int T>
__global__ __launch_bounds__(256) void linear_small_fwd_f32_kernel(SmallLinearFwd p) {
  __shared__ SmallShared<T, 4> sm;
  int const nbn = (p.out_dim + T - 1) / T;
  SmallOperand<true, FFK_ACT_NONE> const a = {p.x, nullptr, p.in_dim, 0}, b = {p.w, nullptr, p.in_dim, 0};
  auto store = [&](int m, int n, float v) {
    v += p.bias != nullptr ? p.bias[n] : 0.0f;
    switch (p.act) {
      case FFK_ACT_RELU: v = v >= 0.0f ? v : 0.0f; break;  // tensor_accessor_unary_ops.cc:32-38 keeps x >= 0
      case FFK_ACT_SIGMOID: v = 1.0f / (1.0f + expf(-v)); break;
      case FFK_ACT_TANH: v = tanhf(v); break;
      case FFK_ACT_GELU: v = gelu_forward(v); break;
      default: break;
    }
    p.y[(int64_t)m * p.out_dim + n] = v;
  };
  small_tile<T, 4, 4>(a, b, p.batch, p.out_dim, p.in_dim, ((int)blockIdx.x / nbn) * T, ((int)blockIdx.x % nbn) * T, true,
                      nullptr, 0, store, false, [](int, float) {}, sm);
}

// The tile (16, 32, or 0: the general kernels) of the one-launch forward.  Measured against the 64x64
// tiles of the general kernel: 512 x 256 -> 512 6.0 us (12.3), 1024 x 512 -> 512 12.6 (19.4); at
// 1024 x 1024 -> 1024 the wave tiles' operand traffic loses, 41 (30).  A few rows over a wide weight
// are bound by reading it and keep these tiles.
static int small_linear_fwd_tile(int64_t batch, int64_t in_dim, int64_t out_dim) {
  if (in_dim > 1024 || batch >= (1 << 20) || out_dim >= (1 << 20)) return 0;
  int64_t const area = batch * out_dim;
  if (area <= 16 * 16 * 1024) return 16;
  if (area <= 32 * 32 * 640 || (batch <= 32 && area <= 32 * 32 * 4096)) return 32;
  return 0;
}
// The tile and the waves a workgroup of the one-launch backward.  A long batch over a small weight has
// few tiles of weight_grad and a long reduction: sixteen waves share a tile there (8000 x 64 -> 64
// 39 us, 860 with one workgroup of four waves a 128 x 64 tile).
struct SmallBwdShape { int tile, waves; };
static SmallBwdShape small_linear_bwd_shape(int dtype, int64_t batch, int64_t in_dim, int64_t out_dim) {
  if (dtype != FFK_FLOAT || batch > 16384 || out_dim > 1024 || in_dim > 16384) return {0, 0};
  int64_t const weights = out_dim * in_dim, both = (batch + out_dim) * in_dim;
  if (batch <= 512 && both <= 16 * 16 * 1024) return {16, 4};
  if (batch > 512 && weights <= 16 * 16 * 256) return {16, 16};
  if (batch <= 1024 && both <= 32 * 32 * 2048) return {32, 4};
  if (batch > 1024 && weights <= 32 * 32 * 256) return {32, 16};
  return {0, 0};
}
template <int T, int WAVES>
static void small_linear_bwd_launch(hipStream_t st, int activation, SmallLinearBwd p) {
  int64_t const nbn = ceil_div(p.in_dim, T);
  p.blocks_dx = (int)ceil_div(ceil_div(p.batch, T) * nbn, WAVES / 4);
  int const blocks = p.blocks_dx + (int)(ceil_div(p.out_dim, T) * nbn);
  switch (activation) {
    case FFK_ACT_RELU: linear_small_bwd_f32_kernel<T, FFK_ACT_RELU, WAVES><<<blocks, WAVES * 64, 0, st>>>(p); break;
    case FFK_ACT_SIGMOID: linear_small_bwd_f32_kernel<T, FFK_ACT_SIGMOID, WAVES><<<blocks, WAVES * 64, 0, st>>>(p); break;
    case FFK_ACT_TANH: linear_small_bwd_f32_kernel<T, FFK_ACT_TANH, WAVES><<<blocks, WAVES * 64, 0, st>>>(p); break;
    default: linear_small_bwd_f32_kernel<T, FFK_ACT_NONE, WAVES><<<blocks, WAVES * 64, 0, st>>>(p); break;
  }
}

}  // namespace ffk

using namespace ffk;

// bf16 gradient rows of no whole 16 bytes (a vocabulary's 50257): the products then could only be
// read an element's address at a time, which costs them half their rate ([2048, 50257] . [50257, 1024]
// 636 us so).  The pass that sums the bias gradient also writes g with rows that are.
static bool linear_pads_grad(int dtype, int64_t out_dim) { return dtype == FFK_BF16 && out_dim % 8 != 0; }
static int64_t linear_grad_ld(int dtype, int64_t out_dim) {
  return linear_pads_grad(dtype, out_dim) ? (out_dim + 63) / 64 * 64 : out_dim;
}

// Room for the partial sums of reductions that are split over workgroups: it lies at the end of the
// workspace, where it overlaps neither g nor column sums that wait there, and it depends on nothing else
// the call asks for, so that each gradient has the same bits whatever becomes of the others (but for a bias
// gradient asked for alone in bf16, whose column sums are a kernel of their own).
// in_dim is not known here; what the splits can use is bounded all the same.
//
// Of the sequence of products, for the input gradient:
//  fp32: 16 x 16 tiles on two workgroups a CU at most, fewer than 1024 tiles of 1 KB (gemm_f32.hip).
//  bf16: one round of 256 x 256 tiles in fp32, 64 MB ([2048, 50257] . [50257, 1024] takes all of it: 8
//  splits, 210 us, 446 without), 16 splits of 2048 columns for few rows.  Shorter reductions, and rows
//  fewer than a tile's, are not split (gemm_splits_for).
static size_t linear_product_split_bytes(int dtype, int64_t batch, int64_t out_dim) {
  if (dtype == FFK_FLOAT) return out_dim >= 2048 ? size_t(1) << 20 : 0;
  if (dtype != FFK_BF16 || out_dim <= 63 * 64 || batch < 128) return 0;
  return batch >= 512 ? size_t(64) << 20 : (size_t)batch << 17;
}
// Of whichever form the backward takes.  The jobs of one launch (linear_any.hip) cut reductions that are long
// enough, for outputs so few that parts of them have to fill the chip: 512 parts of 64 x 64 at 16 KB, and where
// the plan would have more, or larger ones, it makes do.
static size_t linear_split_bytes(int dtype, int64_t batch, int64_t out_dim) {
  size_t const any = dtype == FFK_BF16 && linear_any_may_split(batch, out_dim) ? size_t(8) << 20 : 0;
  return std::max(any, linear_product_split_bytes(dtype, batch, out_dim));
}

// Whether the two tensors share memory.
static bool overlap(void const *a, int64_t a_elems, void const *b, int64_t b_elems, size_t size) {
  uintptr_t const p = reinterpret_cast<uintptr_t>(a), q = reinterpret_cast<uintptr_t>(b);
  return a != nullptr && b != nullptr && p < q + (size_t)b_elems * size && q < p + (size_t)a_elems * size;
}

// Whether the backward runs as the jobs of one launch (linear_any.hip).  aligned: the input and the weight
// can be read 16 bytes at a time, so that the sequence below has the pipelined products, which overtake the
// register-staged ones where there is enough to multiply.  Whole backward, this against the sequence, with
// the forward's share: 7616 x 2176 -> 44 (8046 tiles of 64 deep k's in the two products) 47 and 71 us; 6976 x
// 576 -> 384 (11 772) 57 and 57; 1280 x 2688 -> 768 (20 160) 43 and 43; 4181 x 2560 -> 247 (21 120) 96 and 81;
// 2689 x 1728 -> 1024 114 and 69.  The sequence's tiles are wider than 128 columns: 1537 x 128 -> 48518 229 and
// 265, 832 x 64 -> 41672 109 and 239.
// Other operands gain at all sizes: 57 x 56 -> 64 9 and 21 us, 2944 x 3446 -> 1488 194 and 479.
static bool linear_any_takes(int64_t batch, int64_t in_dim, int64_t out_dim, bool aligned) {
  if (!aligned) return true;
  // whole tiles that fill half the chip: the fused operators of the encoder layer promise the bits of this sequence
  if (batch % 128 == 0 && in_dim % 128 == 0 && out_dim % 64 == 0 && (batch / 128) * (in_dim / 128) >= kNumCU / 2) return false;
  int64_t const k_tiles = ceil_div(batch, 64) * ceil_div(in_dim, 64) * ceil_div(out_dim, 64);
  return k_tiles <= (in_dim <= 128 ? 40000 : 8000);
}

// g and the column sums
static size_t linear_gradient_bytes(int dtype, int activation, int use_bias, int64_t batch, int64_t out_dim) {
  size_t bytes = 0;
  if (activation != FFK_ACT_NONE || linear_pads_grad(dtype, out_dim)) {
    bytes += align256((size_t)batch * (size_t)linear_grad_ld(dtype, out_dim) * dtype_size(dtype));
  }
  if (use_bias) {
    bytes += align256((size_t)colsum_partials_elems(batch, out_dim) * sizeof(float));
  }
  return bytes;
}

extern "C" size_t ffk_linear_backward_workspace_bytes(int dtype, int activation,
                                                      int use_bias,
                                                      int64_t batch,
                                                      int64_t out_dim) {
  return linear_gradient_bytes(dtype, activation, use_bias, batch, out_dim) + linear_split_bytes(dtype, batch, out_dim);
}

extern "C" int ffk_linear_forward(ffk_stream_t stream, int dtype,
                                  int activation, void const *input,
                                  void *output, void const *weight,
                                  void const *bias, int64_t batch,
                                  int64_t in_dim, int64_t out_dim) {
  FFK_REQUIRE(dtype == FFK_FLOAT || dtype == FFK_BF16,
              "linear_forward: dtype %d not supported", dtype);
  FFK_REQUIRE(activation >= FFK_ACT_NONE && activation <= FFK_ACT_GELU,
              "linear_forward: Unhandled activation function %d", activation);
  FFK_REQUIRE(batch > 0 && in_dim > 0 && out_dim > 0,
              "linear_forward: non-positive dimension");
  FFK_REQUIRE(input && output && weight, "linear_forward: NULL tensor");
  int const tile = dtype == FFK_FLOAT ? small_linear_fwd_tile(batch, in_dim, out_dim) : 0;
  if (tile != 0) {
    SmallLinearFwd p = {static_cast<float const *>(input), static_cast<float const *>(weight),
                        static_cast<float const *>(bias), static_cast<float *>(output),
                        (int)batch, (int)in_dim, (int)out_dim, activation};
    unsigned const blocks = (unsigned)(ceil_div(batch, tile) * ceil_div(out_dim, tile));
    if (tile == 16) {
      linear_small_fwd_f32_kernel<16><<<blocks, 256, 0, as_stream(stream)>>>(p);
    } else {
      linear_small_fwd_f32_kernel<32><<<blocks, 256, 0, as_stream(stream)>>>(p);
    }
    FFK_CHECK_LAUNCH();
    return FFK_OK;
  }
  GemmEpilogue ep;
  ep.bias = bias;
  ep.activation = activation;
  // output[batch,out] = input[batch,in] . weight[out,in]^T
  return gemm_dispatch(as_stream(stream), dtype, false, true, batch, out_dim,
                       in_dim, input, in_dim, weight, in_dim, output, out_dim, ep);
}

// input_tail: operators the input gradient passes through while it is written
// (GemmEpilogue's tail fields), or nullptr.
static int linear_backward_impl(
    ffk_stream_t stream, int dtype, int activation, int relu_grad_mode,
    void const *output, void const *output_grad, void const *input,
    void *input_grad, void const *weight, void *weight_grad, void *bias_grad,
    int64_t batch, int64_t in_dim, int64_t out_dim, void *workspace,
    size_t workspace_bytes, int accumulate, GemmEpilogue const *input_tail) {
  FFK_REQUIRE(dtype == FFK_FLOAT || dtype == FFK_BF16,
              "linear_backward: dtype %d not supported", dtype);
  FFK_REQUIRE(activation >= FFK_ACT_NONE && activation <= FFK_ACT_TANH,
              "linear_backward: Unhandled activation function %d (GELU needs "
              "the pre-activation; use an ElementUnary GELU op)",
              activation);
  FFK_REQUIRE(batch > 0 && in_dim > 0 && out_dim > 0,
              "linear_backward: non-positive dimension");
  FFK_REQUIRE(output_grad && weight && input, "linear_backward: NULL tensor");
  hipStream_t st = as_stream(stream);
  if (activation != FFK_ACT_NONE) {
    FFK_REQUIRE(output != nullptr, "linear_backward: output needed for activation");
  }
  // a small fp32 problem whose three gradients are all asked for: one launch, no scratch
  SmallBwdShape const small = input_tail == nullptr && input_grad != nullptr && weight_grad != nullptr
                                  ? small_linear_bwd_shape(dtype, batch, in_dim, out_dim) : SmallBwdShape{0, 0};
  if (small.tile != 0) {
    SmallLinearBwd p = {};
    p.y = static_cast<float const *>(output);
    p.dy = static_cast<float const *>(output_grad);
    p.x = static_cast<float const *>(input);
    p.w = static_cast<float const *>(weight);
    p.dx = static_cast<float *>(input_grad);
    p.dw = static_cast<float *>(weight_grad);
    p.db = static_cast<float *>(bias_grad);
    p.batch = (int)batch;
    p.in_dim = (int)in_dim;
    p.out_dim = (int)out_dim;
    p.relu_mode = relu_grad_mode;
    p.accumulate = accumulate;
    if (small.tile == 16 && small.waves == 16) {
      small_linear_bwd_launch<16, 16>(st, activation, p);
    } else if (small.tile == 16) {
      small_linear_bwd_launch<16, 4>(st, activation, p);
    } else if (small.waves == 16) {
      small_linear_bwd_launch<32, 16>(st, activation, p);
    } else {
      small_linear_bwd_launch<32, 4>(st, activation, p);
    }
    FFK_CHECK_LAUNCH();
    return FFK_OK;
  }
  bool const act = activation != FFK_ACT_NONE;
  bool const sums = bias_grad != nullptr;
  // (asked for whichever kernels run: a caller need not know which of them use it)
  size_t const partial_bytes = sums ? align256((size_t)colsum_partials_elems(batch, out_dim) * sizeof(float)) : 0;
  auto grad_bytes = [&](int64_t ld) { return align256((size_t)batch * (size_t)ld * dtype_size(dtype)); };
  size_t const least = partial_bytes + (act ? grad_bytes(out_dim) : 0);
  if (least > 0 && (workspace == nullptr || workspace_bytes < least)) {
    return fail(FFK_ERR_WORKSPACE, "linear_backward: workspace of %zu bytes needed, %zu given", least, workspace_bytes);
  }
  if (dtype == FFK_BF16 && input_tail == nullptr && std::max(std::max(batch, in_dim), out_dim) < (1 << 30) && (input_grad != nullptr || weight_grad != nullptr) &&
      !tl_layer_operators && option(FFK_OPTION_GEMM_VARIANT) == 0 &&
      linear_any_takes(batch, in_dim, out_dim, in_dim % 8 == 0 && aligned16(weight) && aligned16(input))) {
    size_t const split = linear_split_bytes(dtype, batch, out_dim);
    LinearAnyPlan const plan = linear_any_plan(batch, in_dim, out_dim, split);
    bool const room = plan.scratch == 0 || (workspace != nullptr && aligned16(workspace) && workspace_bytes >= split);
    // one launch reads what it writes elsewhere: a gradient over one of the operands takes the sequence below
    void const *const out[3] = {input_grad, weight_grad, bias_grad};
    int64_t const out_elems[3] = {batch * in_dim, out_dim * in_dim, out_dim};
    void const *const in[4] = {output, output_grad, input, weight};
    int64_t const in_elems[4] = {act ? batch * out_dim : 0, batch * out_dim, batch * in_dim, out_dim * in_dim};
    bool apart = true;
    for (int o = 0; o < 3; o++)
      for (int i = 0; i < 4; i++) apart = apart && !overlap(out[o], out_elems[o], in[i], in_elems[i], 2);
    if (room && apart) {
      // the bias gradient is written here and now: a collected job that writes it comes first
      if (ColreduceBatch *const waiting = tl_colreduce_batch; waiting != nullptr && sums) {
        bool clash = false;
        for (int k = 0; k < waiting->count; k++) clash = clash || waiting->job[k].out0 == bias_grad || waiting->job[k].out1 == bias_grad;
        if (clash) FFK_HIP(colreduce_flush(st, *waiting));
      }
      LinearAnyArgs const a = {static_cast<bf16 const *>(output), static_cast<bf16 const *>(output_grad),
                               static_cast<bf16 const *>(input), static_cast<bf16 const *>(weight),
                               static_cast<bf16 *>(input_grad), static_cast<bf16 *>(weight_grad),
                               static_cast<bf16 *>(bias_grad), (int)batch, (int)in_dim, (int)out_dim, relu_grad_mode,
                               accumulate};
      void *const scratch = plan.scratch == 0 ? nullptr : static_cast<uint8_t *>(workspace) + ((workspace_bytes - split) & ~(size_t)255);
      FFK_HIP(linear_any_backward(st, activation, a, plan, scratch));
      return FFK_OK;
    }
  }
  // rows padded to whole 16 bytes, if the products can read the other operands so and there is a pass
  // over g anyway or the products are large enough to pay for one
  bool pad = linear_pads_grad(dtype, out_dim) && in_dim % 8 == 0 && input_tail == nullptr && aligned16(weight) &&
             aligned16(input) && (input_grad != nullptr || weight_grad != nullptr) &&
             (sums || act || batch * in_dim * out_dim >= (int64_t(1) << 26));
  // (a caller that knows the sizes without padding and splits keeps working)
  if (pad && (workspace == nullptr || !aligned16(workspace) ||
              workspace_bytes < partial_bytes + grad_bytes(linear_grad_ld(dtype, out_dim)))) {
    pad = false;
  }
  uint8_t *ws = static_cast<uint8_t *>(workspace);
  void const *g = output_grad;
  int64_t const ldg = pad ? linear_grad_ld(dtype, out_dim) : out_dim;
  int rc;
  if (act || pad) {
    rc = linear_grad(st, dtype, activation, relu_grad_mode, output, output_grad, ws, ldg, batch, out_dim, bias_grad,
                     (accumulate & FFK_ACC_BIAS) != 0, reinterpret_cast<float *>(ws + grad_bytes(ldg)));
    if (rc != FFK_OK) return rc;
    g = ws;
  }
  GemmEpilogue ep;
  ep.a_padded = pad;
  if (input_grad != nullptr) {
    GemmEpilogue dx = input_tail != nullptr ? *input_tail : ep;
    dx.accumulate = (accumulate & FFK_ACC_INPUT) != 0;
    size_t const used = partial_bytes + (act || pad ? grad_bytes(ldg) : 0), split = linear_product_split_bytes(dtype, batch, out_dim);
    if (input_tail == nullptr && split > 0 && aligned16(workspace) && workspace_bytes >= used + split) {
      dx.splitk_ws = ws + ((workspace_bytes - split) & ~(size_t)255);
      // ... of no more partial sums than there are weights: beyond that it depends (4000 x 20 over 2048 in fp32
      // 20 us unsplit, 23 in two; in bf16 2048 x 696 over 24566 130 us in two, 142 in eight, but 2048 x 432 over
      // 50895 230 us in four, 198 in sixteen)
      dx.splitk_ws_bytes = std::min(split, (size_t)in_dim * (size_t)out_dim * dtype_size(dtype));
    }
    // input_grad[batch,in] = g[batch,out] . weight[out,in]
    if (input_tail != nullptr &&
        !gemm_tail_supported(dtype, false, false, batch, in_dim, out_dim, g, out_dim, weight, in_dim,
                             input_grad, in_dim, dx)) {
      return FFK_ERR_UNSUPPORTED;  // before anything is launched: the caller runs the separate operators
    }
    rc = gemm_dispatch(st, dtype, false, false, batch, in_dim, out_dim, g, ldg, weight, in_dim, input_grad, in_dim, dx);
    if (rc != FFK_OK) return rc;
  }
  if (weight_grad != nullptr) {
    ep.accumulate = (accumulate & FFK_ACC_WEIGHT) != 0;
    // weight_grad[out,in] = g[batch,out]^T . input[batch,in]
    rc = weight_grad_dispatch(st, dtype, out_dim, in_dim, batch, g, ldg, input, in_dim, weight_grad, in_dim, ep);
    if (rc != FFK_OK) return rc;
  }
  if (sums && !act && !pad) {
    rc = colsum_dispatch(st, dtype, g, out_dim, batch, out_dim, bias_grad,
                         (accumulate & FFK_ACC_BIAS) != 0, reinterpret_cast<float *>(ws));
    if (rc != FFK_OK) return rc;
  }
  return FFK_OK;
}

extern "C" int ffk_linear_backward(
    ffk_stream_t stream, int dtype, int activation, int relu_grad_mode,
    void const *output, void const *output_grad, void const *input,
    void *input_grad, void const *weight, void *weight_grad, void *bias_grad,
    int64_t batch, int64_t in_dim, int64_t out_dim, void *workspace,
    size_t workspace_bytes, int accumulate) {
  return linear_backward_impl(stream, dtype, activation, relu_grad_mode, output, output_grad, input,
                              input_grad, weight, weight_grad, bias_grad, batch, in_dim, out_dim,
                              workspace, workspace_bytes, accumulate, nullptr);
}

extern "C" int ffk_linear_l2_regularizer_grad(ffk_stream_t stream, int dtype, void const *weight,
                                              void *weight_grad, int64_t elems, float lambda) {
  FFK_REQUIRE(dtype == FFK_FLOAT || dtype == FFK_BF16, "linear_l2_regularizer_grad: dtype %d not supported", dtype);
  FFK_REQUIRE(weight && weight_grad, "linear_l2_regularizer_grad: NULL tensor");
  FFK_REQUIRE(elems > 0, "linear_l2_regularizer_grad: non-positive element count");
  hipStream_t st = as_stream(stream);
  FFK_HIP(dtype == FFK_FLOAT ? l2_reg_grad<float>(st, weight, weight_grad, elems, lambda)
                             : l2_reg_grad<bf16>(st, weight, weight_grad, elems, lambda));
  return FFK_OK;
}

namespace ffk {

size_t linear_sequence_workspace_bytes(int dtype, int activation, int use_bias, int64_t batch, int64_t out_dim) {
  return linear_gradient_bytes(dtype, activation, use_bias, batch, out_dim) + linear_product_split_bytes(dtype, batch, out_dim);
}

int linear_gelu_dropout_forward(hipStream_t st, int dtype, void const *input, void *output,
                                void *dropped, void const *weight, void const *bias, int64_t batch,
                                int64_t in_dim, int64_t out_dim, float rate, uint64_t seed,
                                uint64_t offset, bool any_size) {
  FFK_REQUIRE(input && output && dropped && weight, "linear_gelu_dropout_forward: NULL tensor");
  FFK_REQUIRE(batch > 0 && in_dim > 0 && out_dim > 0, "linear_gelu_dropout_forward: non-positive dimension");
  GemmEpilogue ep;
  ep.bias = bias;
  ep.tail = GemmEpilogue::kTailGeluDropout;
  ep.tail_any_size = any_size;
  ep.tail_out = dropped;
  int const prc = make_dropout_params("linear_gelu_dropout_forward", rate, seed, offset, ep.tail_dropout);
  if (prc != FFK_OK) return prc;
  if (!gemm_tail_supported(dtype, false, true, batch, out_dim, in_dim, input, in_dim, weight, in_dim,
                           output, out_dim, ep)) {
    return FFK_ERR_UNSUPPORTED;
  }
  return gemm_dispatch(st, dtype, false, true, batch, out_dim, in_dim, input, in_dim, weight, in_dim,
                       output, out_dim, ep);
}

int linear_relu_dropout_forward(hipStream_t st, int dtype, void const *input, void *output, void *dropped,
                                void const *weight, void const *bias, int64_t batch, int64_t in_dim, int64_t out_dim,
                                float rate, uint64_t seed, uint64_t offset) {
  GemmEpilogue ep;
  ep.bias = bias;
  ep.activation = FFK_ACT_RELU;
  ep.tail = GemmEpilogue::kTailActDropout;
  ep.tail_any_size = true;
  ep.tail_out = dropped;
  int const prc = make_dropout_params("linear_relu_dropout_forward", rate, seed, offset, ep.tail_dropout);
  if (prc != FFK_OK) return prc;
  if (!gemm_tail_supported(dtype, false, true, batch, out_dim, in_dim, input, in_dim, weight, in_dim, output, out_dim, ep)) {
    return FFK_ERR_UNSUPPORTED;
  }
  return gemm_dispatch(st, dtype, false, true, batch, out_dim, in_dim, input, in_dim, weight, in_dim, output, out_dim, ep);
}

int linear_dropout_add_forward(hipStream_t st, int dtype, void const *input, void const *residual,
                               void *output, void const *weight, void const *bias, int64_t batch,
                               int64_t in_dim, int64_t out_dim, float rate, uint64_t seed,
                               uint64_t offset, bool any_size) {
  FFK_REQUIRE(input && residual && output && weight, "linear_dropout_add_forward: NULL tensor");
  FFK_REQUIRE(batch > 0 && in_dim > 0 && out_dim > 0, "linear_dropout_add_forward: non-positive dimension");
  GemmEpilogue ep;
  ep.bias = bias;
  ep.tail = GemmEpilogue::kTailDropoutAdd;
  ep.tail_any_size = any_size;
  ep.tail_in = residual;
  int const prc = make_dropout_params("linear_dropout_add_forward", rate, seed, offset, ep.tail_dropout);
  if (prc != FFK_OK) return prc;
  if (!gemm_tail_supported(dtype, false, true, batch, out_dim, in_dim, input, in_dim, weight, in_dim,
                           output, out_dim, ep)) {
    return FFK_ERR_UNSUPPORTED;
  }
  return gemm_dispatch(st, dtype, false, true, batch, out_dim, in_dim, input, in_dim, weight, in_dim,
                       output, out_dim, ep);
}

int linear_backward_dropout_gelu(hipStream_t st, int dtype, void const *output_grad, void const *input,
                                 void const *gelu_input, void *input_grad, void const *weight,
                                 void *weight_grad, void *bias_grad, int64_t batch, int64_t in_dim,
                                 int64_t out_dim, void *workspace, size_t workspace_bytes,
                                 int accumulate, float rate, uint64_t seed, uint64_t offset,
                                 void *input_grad_colsum, float *colsum_partials, bool colsum_accumulate,
                                 bool any_size, bool relu) {
  FFK_REQUIRE(output_grad && input && gelu_input && input_grad && weight,
              "linear_backward_dropout_gelu: NULL tensor");
  FFK_REQUIRE(input_grad_colsum == nullptr || colsum_partials != nullptr,
              "linear_backward_dropout_gelu: column sums need scratch for their partial sums");
  FFK_REQUIRE((accumulate & FFK_ACC_INPUT) == 0,
              "linear_backward_dropout_gelu: the input gradient is stored, not added");
  GemmEpilogue tail;
  tail.tail = relu ? GemmEpilogue::kTailDropoutReluGrad : GemmEpilogue::kTailDropoutGeluGrad;
  tail.tail_any_size = any_size;
  tail.tail_in = gelu_input;
  tail.tail_colsum_partials = input_grad_colsum != nullptr ? colsum_partials : nullptr;
  int const prc = make_dropout_params("linear_backward_dropout_gelu", rate, seed, offset, tail.tail_dropout);
  if (prc != FFK_OK) return prc;
  int const rc = linear_backward_impl(st, dtype, FFK_ACT_NONE, 0, nullptr, output_grad, input, input_grad, weight,
                                      weight_grad, bias_grad, batch, in_dim, out_dim, workspace, workspace_bytes,
                                      accumulate, &tail);
  if (rc != FFK_OK || input_grad_colsum == nullptr) return rc;
  return colsum_finish(st, dtype, colsum_partials, batch, in_dim, input_grad_colsum, colsum_accumulate);
}

int linear_backward_add_residual(hipStream_t st, int dtype, void const *output_grad, void const *input, void const *residual,
                                 void *input_grad, void const *weight, void *weight_grad, void *bias_grad, int64_t batch,
                                 int64_t in_dim, int64_t out_dim, void *workspace, size_t workspace_bytes, int accumulate) {
  GemmEpilogue tail;
  tail.tail = GemmEpilogue::kTailDropoutAdd;  // at a rate of zero
  tail.tail_any_size = true;
  tail.tail_in = residual;
  int const prc = make_dropout_params("linear_backward_add_residual", 0.0f, 0, 0, tail.tail_dropout);
  if (prc != FFK_OK) return prc;
  return linear_backward_impl(st, dtype, FFK_ACT_NONE, 0, nullptr, output_grad, input, input_grad, weight, weight_grad,
                              bias_grad, batch, in_dim, out_dim, workspace, workspace_bytes, accumulate & ~FFK_ACC_INPUT,
                              &tail);
}

}  // namespace ffk

extern "C" int ffk_linear_gelu_dropout_forward(ffk_stream_t stream, int dtype, void const *input,
                                               void *output, void *dropped, void const *weight,
                                               void const *bias, int64_t batch, int64_t in_dim,
                                               int64_t out_dim, float rate, uint64_t seed,
                                               uint64_t offset) {
  int const rc = ffk::linear_gelu_dropout_forward(as_stream(stream), dtype, input, output, dropped, weight,
                                                  bias, batch, in_dim, out_dim, rate, seed, offset);
  if (rc == FFK_ERR_UNSUPPORTED) {
    return fail(FFK_ERR_UNSUPPORTED, "linear_gelu_dropout_forward: no fused kernel for this shape; "
                                     "run Linear, GELU and Dropout one after the other");
  }
  return rc;
}

extern "C" int ffk_linear_dropout_add_forward(ffk_stream_t stream, int dtype, void const *input,
                                              void const *residual, void *output, void const *weight,
                                              void const *bias, int64_t batch, int64_t in_dim,
                                              int64_t out_dim, float rate, uint64_t seed,
                                              uint64_t offset) {
  int const rc = ffk::linear_dropout_add_forward(as_stream(stream), dtype, input, residual, output, weight,
                                                 bias, batch, in_dim, out_dim, rate, seed, offset);
  if (rc == FFK_ERR_UNSUPPORTED) {
    return fail(FFK_ERR_UNSUPPORTED, "linear_dropout_add_forward: no fused kernel for this shape; "
                                     "run Linear, Dropout and the addition one after the other");
  }
  return rc;
}

extern "C" int ffk_linear_backward_dropout_gelu(
    ffk_stream_t stream, int dtype, void const *output_grad, void const *input, void const *gelu_input,
    void *input_grad, void const *weight, void *weight_grad, void *bias_grad, int64_t batch,
    int64_t in_dim, int64_t out_dim, void *workspace, size_t workspace_bytes, int accumulate,
    float rate, uint64_t seed, uint64_t offset) {
  int const rc = ffk::linear_backward_dropout_gelu(as_stream(stream), dtype, output_grad, input, gelu_input,
                                                   input_grad, weight, weight_grad, bias_grad, batch,
                                                   in_dim, out_dim, workspace, workspace_bytes,
                                                   accumulate, rate, seed, offset, nullptr, nullptr, false);
  if (rc == FFK_ERR_UNSUPPORTED) {
    return fail(FFK_ERR_UNSUPPORTED, "linear_backward_dropout_gelu: no fused kernel for this shape; "
                                     "run Linear backward, Dropout backward and GELU backward one after the other");
  }
  return rc;
}

extern "C" size_t ffk_dropout_backward_bias_grad_workspace_bytes(int64_t batch, int64_t out_dim) {
  return align256((size_t)colsum_partials_elems(batch, out_dim) * sizeof(float));
}

extern "C" int ffk_dropout_backward_bias_grad(ffk_stream_t stream, int dtype, void const *output_grad,
                                              void *input_grad, int64_t batch, int64_t out_dim, void *bias_grad,
                                              int accumulate_bias, void *workspace, size_t workspace_bytes,
                                              float rate, uint64_t seed, uint64_t offset) {
  FFK_REQUIRE(output_grad && input_grad && bias_grad, "dropout_backward_bias_grad: NULL tensor");
  FFK_REQUIRE(batch > 0 && out_dim > 0, "dropout_backward_bias_grad: non-positive dimension");
  size_t const need = ffk_dropout_backward_bias_grad_workspace_bytes(batch, out_dim);
  if (workspace == nullptr || workspace_bytes < need) {
    return fail(FFK_ERR_WORKSPACE, "dropout_backward_bias_grad: workspace of %zu bytes needed, %zu given", need,
                workspace_bytes);
  }
  DropoutParams dp;
  int const prc = make_dropout_params("dropout_backward_bias_grad", rate, seed, offset, dp);
  if (prc != FFK_OK) return prc;
  int const rc = dropout_backward_colsum(as_stream(stream), dtype, output_grad, input_grad, batch, out_dim, bias_grad,
                                         accumulate_bias != 0, static_cast<float *>(workspace), dp);
  if (rc == FFK_ERR_UNSUPPORTED) {
    return fail(FFK_ERR_UNSUPPORTED, "dropout_backward_bias_grad: no fused kernel for this shape; run Dropout "
                                     "backward and let the Linear's backward sum its bias gradient");
  }
  return rc;
}

extern "C" int ffk_linear_backward_dropout_gelu_bias_grad(
    ffk_stream_t stream, int dtype, void const *output_grad, void const *input, void const *gelu_input,
    void *input_grad, void const *weight, void *weight_grad, void *bias_grad, int64_t batch, int64_t in_dim,
    int64_t out_dim, void *workspace, size_t workspace_bytes, int accumulate, float rate, uint64_t seed,
    uint64_t offset, void *gelu_bias_grad, int accumulate_gelu_bias, void *gelu_bias_workspace,
    size_t gelu_bias_workspace_bytes) {
  FFK_REQUIRE(gelu_bias_grad != nullptr, "linear_backward_dropout_gelu_bias_grad: NULL bias gradient");
  size_t const need = ffk_dropout_backward_bias_grad_workspace_bytes(batch, in_dim);
  if (gelu_bias_workspace == nullptr || gelu_bias_workspace_bytes < need) {
    return fail(FFK_ERR_WORKSPACE, "linear_backward_dropout_gelu_bias_grad: workspace of %zu bytes needed for the "
                                   "column sums, %zu given", need, gelu_bias_workspace_bytes);
  }
  int const rc = ffk::linear_backward_dropout_gelu(as_stream(stream), dtype, output_grad, input, gelu_input, input_grad,
                                                   weight, weight_grad, bias_grad, batch, in_dim, out_dim, workspace,
                                                   workspace_bytes, accumulate, rate, seed, offset, gelu_bias_grad,
                                                   static_cast<float *>(gelu_bias_workspace), accumulate_gelu_bias != 0);
  if (rc == FFK_ERR_UNSUPPORTED) {
    return fail(FFK_ERR_UNSUPPORTED, "linear_backward_dropout_gelu_bias_grad: no fused kernel for this shape; "
                                     "use ffk_linear_backward_dropout_gelu and let the first Linear's backward sum "
                                     "its bias gradient");
  }
  return rc;
}
