// Tiles of fp32 products whose time is latency, not arithmetic: outputs of few elements, short
// reductions, or long ones over few outputs.  A group of waves owns a T x T tile of the output and
// splits its reduction; every operand element goes from memory straight into the register the MFMA
// takes it from (no LDS, no barrier before the arithmetic), and the partial tiles meet once in LDS.
// A lane supplies the MFMA with one row and one k of each operand; since the sum over k may be taken
// in any order, lane group g takes k = 4 g .. 4 g + 3 of a block of 4 * groups k's, so that an operand
// whose k index is contiguous is read 16 bytes at a time.
#pragma once
#include "ffk_common.h"
#include <type_traits>

namespace ffk {

// An operand's element (r, k): KC: p[r * ld + k]; otherwise p[k * ld + r].  ACT: the element is
// act'(y) * p with y laid out like p (FFK_ACT_NONE: p alone).  ACT is a template argument of the
// kernel: a run-time switch puts a branch and a wait between every two loads of a thread, and the
// kernel's time is its round trips to memory.
template <bool KC, int ACT>
struct SmallOperand {
  float const *p, *y;
  int64_t ld;
  int mode;
  static constexpr bool kPair = ACT != FFK_ACT_NONE;
  // what a lane holds of one block of k's: nothing is computed from it before the MFMAs (arithmetic
  // on a loaded value any earlier would make the wave wait for the load it is meant to run under)
  struct Raw {
    f32x4 v, y;
  };
  __device__ __forceinline__ static f32x4 four(float const *q, int64_t ld, int r, int k, int last, bool whole) {
    f32x4 v;
    if (whole) {
      if constexpr (KC) return __builtin_bit_cast(f32x4, load_raw_any(q + (int64_t)r * ld + k));
#pragma unroll
      for (int j = 0; j < 4; j++) v[j] = q[(int64_t)(k + j) * ld + r];
    } else {  // k's past the last one are read from it (and count as zeros)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        int const kk = k + j < last ? k + j : last;
        v[j] = KC ? q[(int64_t)r * ld + kk] : q[(int64_t)kk * ld + r];
      }
    }
    return v;
  }
  __device__ __forceinline__ void fetch(Raw &raw, int r, int k, int last, bool whole) const {
    raw.v = four(p, ld, r, k, last, whole);
    if constexpr (kPair) raw.y = four(y, ld, r, k, last, whole);
  }
  __device__ __forceinline__ float value(Raw const &raw, int j) const {
    return activation_grad<ACT>(mode, kPair ? raw.y[j] : 0.0f, raw.v[j]);
  }
};

template <int T>
struct SmallAcc {
  typedef float type __attribute__((ext_vector_type(T * T / 64)));
};
template <int T, int WAVES>
struct SmallShared {
  float acc[WAVES][T * T];
  float bias[WAVES][T];
};

// S waves of the workgroup's WAVES work on one tile (each on its part of the reduction), so a
// workgroup holds WAVES / S tiles; this wave is number `part` of the S and works on tile `slot`.
// live: the slot holds a tile (the last workgroup's spare slots do not).
// The T x T tile at (m0, n0) of sum_k a(m, k) * b(n, k), k in [0, K), handed element by element to
// store(m, n, value); rows and columns past the edge are read from the last ones and not stored.
// prior: the tensor the result is added to (accumulating), or NULL.  bias: also store_bias(m, sum_k a(m, k)).
template <int T, int S, int WAVES, typename OA, typename OB, typename FS, typename FB>
__device__ __forceinline__ void small_tile(OA const &a, OB const &b, int M, int N, int K, int m0, int n0, bool live,
                                           float const *prior, int64_t prior_ld, FS store, bool bias, FB store_bias,
                                           SmallShared<T, WAVES> &sm) {
  constexpr int G = 64 / T;        // lane groups
  constexpr int SUB = 4 * G;       // k's of one block
  constexpr int NSUB = 4;          // blocks fetched together
  constexpr int NR = T * T / 64;   // accumulator registers
  int const lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int const part = wave % S, slot0 = wave - part;  // slot0: the first wave of this tile
  int const l = lane % T, g = lane / T;
  int const am = min(m0 + l, M - 1), bn = min(n0 + l, N - 1);
  int const per_wave = (K + S * SUB - 1) / (S * SUB) * SUB;
  int const k_first = part * per_wave, k_end = live ? min(K, k_first + per_wave) : 0;
  typename SmallAcc<T>::type acc;
#pragma unroll
  for (int r = 0; r < NR; r++) acc[r] = 0.0f;
  float bsum = 0.0f;
  typename OA::Raw ra[2][NSUB];
  typename OB::Raw rb[2][NSUB];
  constexpr int CH = NSUB * SUB;
  // ALL: the whole chunk lies below k_end; no branches then, whose joins would make the waves wait
  // for every load in flight
  auto fetch = [&](auto set, auto all, int k0) {
#pragma unroll
    for (int s = 0; s < NSUB; s++) {
      int const k = k0 + s * SUB;
      if (!all.value && k >= k_end) break;  // uniform over the wave, like the choice of the access
      bool const whole = all.value || k + SUB <= k_end;
      a.fetch(ra[set.value][s], am, k + 4 * g, K - 1, whole);
      b.fetch(rb[set.value][s], bn, k + 4 * g, K - 1, whole);
    }
  };
  auto multiply = [&](auto set, auto all, int k0) {
#pragma unroll
    for (int s = 0; s < NSUB; s++) {
      int const k = k0 + s * SUB;
      if (!all.value && k >= k_end) break;
      bool const whole = all.value || k + SUB <= k_end;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        bool const in = whole || k + 4 * g + j < k_end;
        float const av = in ? a.value(ra[set.value][s], j) : 0.0f;
        float const bv = in ? b.value(rb[set.value][s], j) : 0.0f;
        if constexpr (T == 16) {
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av, bv, acc, 0, 0, 0);
        } else {
          acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av, bv, acc, 0, 0, 0);
        }
        bsum += av;
      }
    }
  };
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;
  using Whole = std::true_type;
  using Any = std::false_type;
  int k0 = k_first;
  if (k0 + CH <= k_end) {
    fetch(S0{}, Whole{}, k0);
    while (true) {  // the next chunk is on its way while this one is multiplied (past the last one: this one again)
      fetch(S1{}, Whole{}, k0 + 2 * CH <= k_end ? k0 + CH : k0);
      multiply(S0{}, Whole{}, k0);
      k0 += CH;
      if (k0 + CH > k_end) break;
      fetch(S0{}, Whole{}, k0 + 2 * CH <= k_end ? k0 + CH : k0);
      multiply(S1{}, Whole{}, k0);
      k0 += CH;
      if (k0 + CH > k_end) break;
    }
  }
  if (k0 < k_end) {
    fetch(S0{}, Any{}, k0);
    multiply(S0{}, Any{}, k0);
  }
  // the S partial tiles: of the tile's NR * 64 elements, S * 64 a time
#pragma unroll
  for (int r = 0; r < NR; r++) sm.acc[wave][r * 64 + lane] = acc[r];
  if (bias) {
    if constexpr (T == 16) {
      auto const h = __builtin_amdgcn_permlane16_swap(__float_as_uint(bsum), __float_as_uint(bsum), false, false);
      bsum = __uint_as_float(h[0]) + __uint_as_float(h[1]);
    }
    auto const h = __builtin_amdgcn_permlane32_swap(__float_as_uint(bsum), __float_as_uint(bsum), false, false);
    bsum = __uint_as_float(h[0]) + __uint_as_float(h[1]);
    if (lane < T) sm.bias[wave][lane] = bsum;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < (NR + S - 1) / S; q++) {
    int const r = part + q * S;
    if (NR % S != 0 && r >= NR) break;
    int const at = r * 64 + lane;
    float v = 0.0f;
#pragma unroll
    for (int w = 0; w < S; w += 4) {
      v += (sm.acc[slot0 + w][at] + sm.acc[slot0 + w + 1][at]) + (sm.acc[slot0 + w + 2][at] + sm.acc[slot0 + w + 3][at]);
    }
    int const row = T == 16 ? 4 * g + r : 8 * (r >> 2) + 4 * g + (r & 3);
    int const m = m0 + row, n = n0 + l;
    if (live && m < M && n < N) store(m, n, prior != nullptr ? prior[(int64_t)m * prior_ld + n] + v : v);
  }
  if (bias && part == 0 && lane < T && live && m0 + lane < M) {
    float v = 0.0f;
#pragma unroll
    for (int w = 0; w < S; w += 4) {
      v += (sm.bias[slot0 + w][lane] + sm.bias[slot0 + w + 1][lane]) + (sm.bias[slot0 + w + 2][lane] + sm.bias[slot0 + w + 3][lane]);
    }
    store_bias(m0 + lane, v);
  }
}


}  // namespace ffk
