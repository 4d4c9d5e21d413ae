// Tiles of bf16 products whose operands lie at any address with any row stride (an odd row length, a
// view that begins anywhere): what the direct global->LDS loads of gemm_bf16.h cannot take.
//
// A workgroup of NT threads computes a BM x BN tile.  Operands go through registers, 16 bytes at a time
// at whatever alignment, two k-tiles ahead of the one that is multiplied, into two LDS buffers; a k-tile
// costs one barrier.  No load is guarded: where 16 bytes would pass the end of a row the load begins early
// enough to end with it, and the elements that do not belong are shifted out on the way to LDS, which only
// the workgroups at an edge and the last k-tile do.  (Guarded element loads there made such a workgroup's
// k-tile 2.4 us of branches and round trips: [305, 40606] . [40606, 245] 1523 us.)
// Bound by the LDS reads and the unaligned loads: [4096, 4095] . [4095, 4095] 205 us on 128x128 tiles, 2.8 times
// a product of aligned rows; 243 us with both operands K-contiguous and 436 with neither, one k-tile ahead and
// with guarded edges.  Eight waves of 64x32 a tile and two workgroups a CU (with rows padded by 16 elements;
// by 32 only one fits): four waves of 64x64 take 218-230 us, more k-tiles ahead gain nothing.
//
// An operand can be a product of two tensors read side by side, act'(y) * p: the gradient before a
// Linear's activation, rounded as it would be stored.
#pragma once
#include "gemm.h"
#include "ffk_common.h"

namespace ffk {

constexpr int kBK = 64;        // K extent of one LDS tile
constexpr int kPadK = 8;       // row padding (elements) of a K-contiguous tile
constexpr int kPadMN = 16;     // row padding of an M/N-contiguous tile

// v without its first s elements, zeros behind them.
__device__ __forceinline__ u32x4 drop_elements(u32x4 v, int s) {
  if (s & 4) v = u32x4{v[2], v[3], 0u, 0u};
  if (s & 2) v = u32x4{v[1], v[2], v[3], 0u};
  if (s & 1) {
    v = u32x4{(v[0] >> 16) | (v[1] << 16), (v[1] >> 16) | (v[2] << 16), (v[2] >> 16) | (v[3] << 16), v[3] >> 16};
  }
  return s >= 8 ? u32x4{0u, 0u, 0u, 0u} : v;
}

// Element (r, k) of an operand: KC: p[r * ld + k], otherwise p[k * ld + r]; ROWS rows of it from r0 on.
template <int ROWS, int NT, bool KC, int ACT>
struct AnyOperand {
  static constexpr int kChunks = ROWS * kBK / 8 / NT;  // 16-byte pieces of a thread and k-tile
  static constexpr int kStride = KC ? kBK + kPadK : ROWS + kPadMN;
  static constexpr int kElems = KC ? ROWS * kStride : kBK * kStride;
  static constexpr bool kPair = ACT != FFK_ACT_NONE;
  static_assert(ROWS * kBK / 8 % NT == 0 && NT % (ROWS / 8) == 0 && NT % 8 == 0, "whole pieces, columns that stay");
  struct Raw {
    u32x4 v[kChunks], y[kPair ? kChunks : 1];
  };
  bf16 const *p, *y;
  int64_t ld;
  int R, K, mode;
  int r0, t;
  // KC: the thread's k of every k-tile; otherwise its first row, and the row it loads from instead
  // where 8 of them do not exist there
  int at, from;
  bool edge;  // of the workgroup: some rows of the tile do not exist

  __device__ __forceinline__ void init(bf16 const *p_, bf16 const *y_, int64_t ld_, int R_, int K_, int mode_, int r0_, int t_) {
    p = p_, y = y_, ld = ld_, R = R_, K = K_, mode = mode_, r0 = r0_, t = t_;
    edge = r0 + ROWS > R;
    at = KC ? (t & 7) * 8 : r0 + (t % (ROWS / 8)) * 8;
    from = KC ? 0 : max(0, min(at, R - 8));
  }
  __device__ __forceinline__ int row_of(int i) const { return KC ? (t + i * NT) >> 3 : (t + i * NT) / (ROWS / 8); }
  __device__ __forceinline__ int64_t offset(int i, int k0, bool tail) const {
    if constexpr (KC) {
      return (int64_t)min(r0 + row_of(i), R - 1) * ld + (tail ? max(0, min(k0 + at, K - 8)) : k0 + at);
    } else {
      int const k = k0 + row_of(i);
      return (int64_t)(tail ? min(k, K - 1) : k) * ld + from;
    }
  }
  // (tail: the k-tile is the last one of the whole reduction and not a whole one)
  __device__ __forceinline__ void fetch(Raw &raw, int k0, bool tail) const {
    int const len = KC ? K : R;  // of the contiguous index; 8 and more but for the smallest products
    bool const tiny = len < 8;
#pragma unroll
    for (int i = 0; i < kChunks; i++) {
      int64_t const o = offset(i, k0, tail);
      raw.v[i] = tiny ? load_raw_first(p + o, len) : load_raw_any(p + o);
      if constexpr (kPair) raw.y[i] = tiny ? load_raw_first(y + o, len) : load_raw_any(y + o);
    }
  }
  // what of piece i belongs to the tile, with the activation's gradient applied
  __device__ __forceinline__ u32x4 value(Raw const &raw, int i, int k0, bool tail) const {
    u32x4 v = raw.v[i];
    if constexpr (kPair) {
      float g[8], out[8];
      unpack_raw(v, g, (bf16 const *)nullptr);
      unpack_raw(raw.y[i], out, (bf16 const *)nullptr);
#pragma unroll
      for (int e = 0; e < 8; e++) g[e] = activation_grad<ACT>(mode, out[e], g[e]);
      v = pack_raw(g, (bf16 const *)nullptr);
    }
    if constexpr (KC) {
      if (tail) v = drop_elements(v, k0 + at - max(0, min(k0 + at, K - 8)));
    } else {
      if (edge) v = drop_elements(v, at - from);
      if (tail && k0 + row_of(i) >= K) v = u32x4{0u, 0u, 0u, 0u};
    }
    return v;
  }
  __device__ __forceinline__ int lds_index(int i) const {
    return KC ? row_of(i) * kStride + (t & 7) * 8 : row_of(i) * kStride + (t % (ROWS / 8)) * 8;
  }
};

// Operand fragment for one 32-row MFMA tile and one 16-wide k step of an LDS tile: lane l supplies row
// l % 32, k = 8 * (l / 32) .. + 7.
template <bool KC>
__device__ __forceinline__ bf16x8 any_fragment(bf16 const *tile, int stride, int row0, int kk, int lane) {
  if constexpr (KC) {
    return *reinterpret_cast<bf16x8 const *>(tile + (row0 + (lane & 31)) * stride + kk * 16 + (lane >> 5) * 8);
  } else {
    // Transposing load: within each 16-lane group, lane i points at 4 elements
    // of row k_(i/4), columns 4*(i%4)..+3, and receives column i of the four
    // rows.  Two loads give 8 consecutive k for this lane's row.
    int const i16 = lane & 15;
    int const col = row0 + ((lane >> 4) & 1) * 16 + (i16 & 3) * 4;
    int const kbase = kk * 16 + (lane >> 5) * 8 + (i16 >> 2);
    typedef s16x4 __attribute__((address_space(3))) * lds_s16x4_ptr;
    union {
      s16x4 h[2];
      bf16x8 v;
    } u;
    u.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(tile + kbase * stride + col));
    u.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(tile + (kbase + 4) * stride + col));
    return u.v;
  }
}

template <int BM, int BN, int WM, int WN, bool KCA, bool KCB, int ACT = FFK_ACT_NONE>
struct AnyTile {
  static constexpr int NT = (BM / WM) * (BN / WN) * 64;
  static constexpr int TM = WM / 32, TN = WN / 32;
  using OpA = AnyOperand<BM, NT, KCA, ACT>;
  using OpB = AnyOperand<BN, NT, KCB, FFK_ACT_NONE>;
  static constexpr int kBufElems = OpA::kElems + OpB::kElems;
  static constexpr size_t kLds = 2 * (size_t)kBufElems * sizeof(bf16);

  f32x16 acc[TM][TN];
  float sums[8];  // SUMS: of A's rows at, at + 1, ... over the reduction

  // k-tiles [kt0, kt1) of the reduction.  smem: kBufElems * 2 elements.
  template <bool SUMS>
  __device__ __forceinline__ void reduce(OpA const &a, OpB const &b, int K, int kt0, int kt1, bf16 *smem) {
    int const lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int const wm0 = (wave / (BN / WN)) * WM, wn0 = (wave % (BN / WN)) * WN;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; e++) sums[e] = 0.0f;
    typename OpA::Raw ra[2];
    typename OpB::Raw rb[2];
    auto fetch = [&](auto slot, int kt) __attribute__((always_inline)) {
      constexpr int S = decltype(slot)::value;
      bool const tail = (kt + 1) * kBK > K;
      a.fetch(ra[S], kt * kBK, tail);
      b.fetch(rb[S], kt * kBK, tail);
    };
    auto put = [&](auto slot, int kt) __attribute__((always_inline)) {
      constexpr int S = decltype(slot)::value;
      bf16 *const as = smem + S * kBufElems, *const bs = as + OpA::kElems;
      bool const tail = (kt + 1) * kBK > K;
#pragma unroll
      for (int i = 0; i < OpA::kChunks; i++) {
        u32x4 const v = a.value(ra[S], i, kt * kBK, tail);
        *reinterpret_cast<u32x4 *>(as + a.lds_index(i)) = v;
        if constexpr (SUMS) {
          float f[8];
          unpack_raw(v, f, (bf16 const *)nullptr);
#pragma unroll
          for (int e = 0; e < 8; e++) sums[e] += f[e];
        }
      }
#pragma unroll
      for (int i = 0; i < OpB::kChunks; i++) {
        *reinterpret_cast<u32x4 *>(bs + b.lds_index(i)) = b.value(rb[S], i, kt * kBK, tail);
      }
    };
    auto step = [&](auto slot, int kt) __attribute__((always_inline)) {
      constexpr int S = decltype(slot)::value;
      __syncthreads();  // tile kt is in LDS, and nobody reads tile kt - 1 any more
      if (kt + 2 < kt1) fetch(slot, kt + 2);
      bf16 const *const as = smem + S * kBufElems, *const bs = as + OpA::kElems;
#pragma unroll
      for (int kk = 0; kk < kBK / 16; kk++) {
        bf16x8 af[TM], bfr[TN];
#pragma unroll
        for (int i = 0; i < TM; i++) af[i] = any_fragment<KCA>(as, OpA::kStride, wm0 + i * 32, kk, lane);
#pragma unroll
        for (int j = 0; j < TN; j++) bfr[j] = any_fragment<KCB>(bs, OpB::kStride, wn0 + j * 32, kk, lane);
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
          for (int j = 0; j < TN; j++)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[i], bfr[j], acc[i][j], 0, 0, 0);
      }
      if (kt + 1 < kt1) put(std::integral_constant<int, S ^ 1>{}, kt + 1);
    };
    using S0 = std::integral_constant<int, 0>;
    using S1 = std::integral_constant<int, 1>;
    fetch(S0{}, kt0);
    if (kt0 + 1 < kt1) fetch(S1{}, kt0 + 1);
    put(S0{}, kt0);
    for (int kt = kt0; kt < kt1; kt += 2) {
      step(S0{}, kt);
      if (kt + 1 < kt1) step(S1{}, kt + 1);
        }
  }

  // f(m, n, value) for every element of the tile that exists: element r of a lane is row
  // 8*(r/4) + 4*(l/32) + r%4, column l % 32 of its 32x32 tile.
  template <typename F>
  __device__ __forceinline__ void store(int m0, int n0, int M, int N, F f) const {
    int const lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int const wm0 = m0 + (wave / (BN / WN)) * WM, wn0 = n0 + (wave % (BN / WN)) * WN;
#pragma unroll
    for (int j = 0; j < TN; j++) {
      int const n = wn0 + j * 32 + (lane & 31);
      if (n >= N) continue;
#pragma unroll
      for (int i = 0; i < TM; i++) {
#pragma unroll
        for (int r = 0; r < 16; r++) {
          int const m = wm0 + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
          if (m < M) f(m, n, acc[i][j][r]);
        }
      }
    }
  }

  // f(m, sum over the reduction of A's row m) for the rows of the tile that exist (A not KC).
  template <typename F>
  __device__ __forceinline__ void store_sums(int m0, int M, bf16 *smem, F f) const {
    static_assert(!KCA, "a thread's pieces have the same rows");
    constexpr int G = BM / 8, P = NT / G;  // groups of rows, threads of a group
    float *const red = reinterpret_cast<float *>(smem);
    static_assert(P * BM * sizeof(float) <= kLds, "room for the threads' sums");
    int const t = threadIdx.x;
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 8; e++) red[(t / G) * BM + (t % G) * 8 + e] = sums[e];
    __syncthreads();
    if (t < BM && m0 + t < M) {
      float s = 0.0f;
      for (int q = 0; q < P; q++) s += red[q * BM + t];
      f(m0 + t, s);
    }
  }
};

}  // namespace ffk
