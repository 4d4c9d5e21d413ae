// Scatter-add of an embedding's gradient where the lookups are few: one launch, no sort.
//
// Every workgroup reads all ids into LDS, a wave takes one lookup and compares its id with all of them, 256 at
// a time.  A row of up to kMatchRun lookups is the wave's that has the first of them: it sums their gradient
// rows, up to 64 / LPR at once, and adds the sum to the weight-gradient row.  Of a row of more lookups the first
// in each 256 sums what those 256 hold and adds it with atomics.  A wave whose lookup is not the first of its
// 256 is done after one comparison; the popular ids, of which most such lookups are, would be found all over.
// The sort and the walk over what it leaves are chains of launches and round trips to memory that do not
// shorten with the number of lookups (2195 of them, 16 floats a row, 9.7 + 8.2 us, 7.1 so; 8000, 128 floats,
// 28 and 15), while n * n comparisons, 64 an instruction, are few for the thousands of lookups this is for.
// (A wave that counts all lookups before its own, and sums every kMatchRun-th and the ones behind it: 31 us.)
#pragma once
#include "ffk_common.h"
#include <type_traits>

namespace ffk {

constexpr int kMatchMax = 8192;
constexpr int kMatchThreads = 1024, kMatchWaves = kMatchThreads / 64;
constexpr int kMatchRun = 32;  // lookups of one id that one wave sums across the 256s
constexpr uint32_t kMatchNone = 0xffffffffu;  // no row

// blockIdx.y: 4 * LPR * G columns.
template <typename IT, typename GT, int LPR, int G>
__global__ __launch_bounds__(kMatchThreads, 8) void embedding_bwd_match_kernel(IT const *__restrict__ idx, GT const *__restrict__ dY,
                                                                              float *dW, int n, FastDiv by_bag, int dim,
                                                                              int64_t num_entries, float scale) {
  constexpr int R = 64 / LPR, U = 4;  // rows at once, and in flight behind each other
  __shared__ __attribute__((aligned(16))) uint32_t ks[kMatchMax];
  __shared__ uint32_t lists[kMatchWaves][256];
  int const t = threadIdx.x, lane = t & 63;
  int const wave = __builtin_amdgcn_readfirstlane(t >> 6);
  int const whole = (n + 1023) & ~1023;
#pragma unroll 4
  for (int i = t; i < whole; i += kMatchThreads) {
    int64_t const id = i < n ? (int64_t)idx[i] : -1;
    ks[i] = (uint64_t)id < (uint64_t)num_entries ? (uint32_t)id : kMatchNone;
  }
  __syncthreads();
  int const p = (int)blockIdx.x * kMatchWaves + wave;
  if (p >= n) return;
  uint32_t const id = __builtin_amdgcn_readfirstlane(ks[p]);
  if (id == kMatchNone) return;
  u32x4 const *const quads = reinterpret_cast<u32x4 const *>(ks) + lane;
  uint32_t *const list = lists[wave];
  // appends the lookups of the 256 from c on that are the row's to the list, returns how many they are
  auto append = [&](u32x4 v, int c, int at) __attribute__((always_inline)) {
    int found = 0, to = at;
    bool same[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
      same[e] = v[e] == id;
      uint64_t const b = __ballot(same[e]);
      to += (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0));
      found += (int)__popcll(b);
    }
#pragma unroll
    for (int e = 0; e < 4; e++) {
      if (same[e]) {
        if (to < 256) list[to] = by_bag.div((uint32_t)(c + 4 * lane + e));
        to++;
      }
    }
    return found;
  };
  int const mine = p & ~255;  // the 256 that p is among
  int own;                    // the row's lookups there; p has to be the first
  {
    u32x4 const v = quads[mine >> 2];
    bool earlier = false;
#pragma unroll
    for (int e = 0; e < 4; e++) earlier |= v[e] == id && mine + 4 * lane + e < p;
    if (__ballot(earlier) != 0) return;
    own = append(v, mine, 0);
  }
  int before = 0, m = own;  // the row's lookups before the own 256; from there on
  for (int turn = 0; turn < 2 && before + m <= kMatchRun; turn++) {
    int const end = turn == 0 ? whole : mine;
    for (int c0 = turn == 0 ? mine + 256 : 0; c0 < end && before + m <= kMatchRun; c0 += 1024) {
      u32x4 v[4];
#pragma unroll
      for (int u = 0; u < 4; u++) v[u] = quads[min(c0 + u * 256, whole - 256) >> 2];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        int const c = c0 + u * 256;
        if (c >= end || __ballot(v[u][0] == id || v[u][1] == id || v[u][2] == id || v[u][3] == id) == 0) continue;
        if (turn == 0) m += append(v[u], c, m);
        else before += append(v[u], c, 256);
      }
    }
  }
  bool const shared = before + m > kMatchRun;  // too many for one wave: each 256's first takes theirs
  if (!shared && before > 0) return;           // the row's first lookup takes all of them
  int const mk = shared ? own : m;
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();

  int const g = lane / LPR, l = lane % LPR;
  int const col0 = (int)blockIdx.y * (G * LPR * 4) + l * 4;
  float *const row_w = dW + (int64_t)id * dim;
  f32x4 old[G], acc[G];
#pragma unroll
  for (int x = 0; x < G; x++) {
    acc[x] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    int const col = col0 + x * LPR * 4;
    if (!shared && g == 0 && col < dim) old[x] = *reinterpret_cast<f32x4 const *>(row_w + col);
  }
  using Raw = typename std::conditional<sizeof(GT) == 2, u32x2, u32x4>::type;
  auto some = [&](int i, auto depth) __attribute__((always_inline)) {
    constexpr int D = decltype(depth)::value;
    Raw raw[D][G];
#pragma unroll
    for (int u = 0; u < D; u++) {
      GT const *const row = dY + (int64_t)list[min(i + u * R + g, mk - 1)] * dim;
#pragma unroll
      for (int x = 0; x < G; x++) raw[u][x] = *reinterpret_cast<Raw const *>(row + min(col0 + x * LPR * 4, dim - 4));
    }
#pragma unroll
    for (int u = 0; u < D; u++) {
      bool const there = i + u * R + g < mk;
#pragma unroll
      for (int x = 0; x < G; x++) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
          float v;
          if constexpr (sizeof(GT) == 2) v = __uint_as_float((e & 1) == 0 ? raw[u][x][e >> 1] << 16 : raw[u][x][e >> 1] & 0xffff0000u);
          else v = __uint_as_float(raw[u][x][e]);
          acc[x][e] += there ? v : 0.0f;
        }
      }
    }
  };
  if (mk <= R) {
    some(0, std::integral_constant<int, 1>{});
  } else {
    for (int i = 0; i < mk; i += R * U) some(i, std::integral_constant<int, U>{});
  }
#pragma unroll
  for (int x = 0; x < G; x++) {
    int const col = col0 + x * LPR * 4;
#pragma unroll
    for (int e = 0; e < 4; e++) {
#pragma unroll
      for (int off = LPR; off < 64; off <<= 1) acc[x][e] += __shfl_xor(acc[x][e], off, 64);
    }
    if (g == 0 && col < dim) {
      if (shared) {
#pragma unroll
        for (int e = 0; e < 4; e++) atomicAdd(row_w + col + e, acc[x][e] * scale);
      } else {
        *reinterpret_cast<f32x4 *>(row_w + col) = f32x4{old[x][0] + acc[x][0] * scale, old[x][1] + acc[x][1] * scale,
                                                        old[x][2] + acc[x][2] * scale, old[x][3] + acc[x][3] * scale};
      }
    }
  }
}

// Where the comparisons, which every 512 columns make anew, are fewer than so many waves' ([lookups, dim], bf16,
// gathered and scattered: 4096 x 1024 17.4 us and 21.9 by the sort, 8192 x 1024 28 either way; fp32, 8192 x 256
// 18.7 and 25.7, 16 000 x 256 41 and 30).
static inline bool embedding_match_takes(int64_t n, int64_t dim, int64_t num_entries) {
  return n * ceil_div(dim, 512) <= kMatchMax && num_entries < (int64_t)kMatchNone;
}

// dim % 4 == 0, both tensors 16-byte aligned, embedding_match_takes; nothing else adds to dw meanwhile.
template <typename IT, typename GT>
static hipError_t embedding_match(hipStream_t st, IT const *idx, GT const *dy, float *dw, int n, int bag, int dim,
                                  int64_t num_entries, float scale) {
  FastDiv const by_bag = make_fast_div((uint32_t)bag);
#define FFK_EMB_MATCH(LPR_, G_)                                                                                     \
  embedding_bwd_match_kernel<IT, GT, LPR_, G_>                                                                      \
      <<<dim3((unsigned)ceil_div(n, kMatchWaves), (unsigned)ceil_div(dim, 4 * LPR_ * G_)), kMatchThreads, 0, st>>>( \
          idx, dy, dw, n, by_bag, dim, num_entries, scale)
  if (dim > 256) FFK_EMB_MATCH(64, 2);
  else if (dim > 128) FFK_EMB_MATCH(64, 1);
  else if (dim > 64) FFK_EMB_MATCH(32, 1);
  else if (dim > 32) FFK_EMB_MATCH(16, 1);
  else if (dim > 16) FFK_EMB_MATCH(8, 1);
  else FFK_EMB_MATCH(4, 1);
#undef FFK_EMB_MATCH
  return hipGetLastError();
}

}  // namespace ffk
