// Embedding gather (forward) and scatter-add (backward) for gfx950.
//
// forward : output[b,:] = sum_j weight[indices[b,j],:], 16 bytes per lane per
//           row access, the index of a bag entry read once per lane group and
//           int64 offsets throughout (the reference does one element per
//           thread with `int` offsets and re-reads the index per element,
//           lib/kernels/src/cuda/embedding_kernels.cu:48-125).
// backward: weight_grad[indices[b,j],:] += output_grad[b,:]: few lookups by one launch that compares all
//           ids (embedding_match.h), more of them sorted by row (radix_sort.h) and walked
//           (embedding_walk.h), and for a caller without the scratch memory, or where rows are no whole
//           16 bytes, with hardware fp32 atomics, one wave instruction covering 64 consecutive floats of
//           a row (reference: atomicAdd per element, embedding_kernels.cu:128-317).
// Indices outside [0, num_entries) are skipped (the reference reads or writes
// out of bounds for them).
#include "ffk_common.h"
#include "embedding_walk.h"
#include "embedding_match.h"
#include "radix_sort.h"
#include <algorithm>
#include <cstdlib>
#include <type_traits>
#include <cstring>

namespace ffk {

constexpr int kEmbThreads = 256;

template <typename OT, int V>
__device__ __forceinline__ void store_out(OT *p, float const (&v)[V]);

template <>
__device__ __forceinline__ void store_out<float, 4>(float *p, float const (&v)[4]) {
  *reinterpret_cast<f32x4 *>(p) = f32x4{v[0], v[1], v[2], v[3]};
}
template <>
__device__ __forceinline__ void store_out<float, 8>(float *p, float const (&v)[8]) {
  *reinterpret_cast<f32x4 *>(p) = f32x4{v[0], v[1], v[2], v[3]};
  *reinterpret_cast<f32x4 *>(p + 4) = f32x4{v[4], v[5], v[6], v[7]};
}
template <>
__device__ __forceinline__ void store_out<bf16, 4>(bf16 *p, float const (&v)[4]) {
  __builtin_nontemporal_store(u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])}, reinterpret_cast<u32x2 *>(p));
}
template <>
__device__ __forceinline__ void store_out<bf16, 8>(bf16 *p, float const (&v)[8]) {
  VecIO<bf16>::store_stream(p, v);
}

// V elements of a table row as floats: 16-byte loads
template <typename WT, int V>
__device__ __forceinline__ void load_row(WT const *p, float (&v)[V]) {
  if constexpr (sizeof(WT) == 4 && V == 8) {
    float a[4], b[4];
    VecIO<float>::load(p, a);
    VecIO<float>::load(p + 4, b);
#pragma unroll
    for (int e = 0; e < 4; e++) {
      v[e] = a[e];
      v[4 + e] = b[e];
    }
  } else {
    static_assert(V == VecIO<WT>::kVec, "one 16-byte load");
    VecIO<WT>::load(p, v);
  }
}
// elements per thread: what makes the store 16 bytes (8 for a bf16 output), at least one 16-byte load
template <typename WT, typename OT>
constexpr int emb_vec() {
  return sizeof(OT) == 2 ? 8 : VecIO<WT>::kVec;
}

// One thread per (bag, 16-byte vector of the row).  BIG: 2^31 and more threads' worth of
// work, 64-bit index arithmetic; otherwise 32-bit with the division by nvec as a multiplication
// (the 64-bit division alone was 130 of the 250 instructions a thread of the plain gather ran,
// and made that kernel bound by the vector ALU).
// CHUNKED: the kernel for bags of eight entries and more (its row buffers cost the plain
// gather half its waves per CU, so single lookups run the instantiation without them).
template <typename IT, typename WT, typename OT, bool BIG, bool CHUNKED>
__global__ __launch_bounds__(kEmbThreads) void embedding_fwd_vec_kernel(
    IT const *__restrict__ idx, OT *__restrict__ out, WT const *__restrict__ W,
    int64_t num_bags, int bag, int nvec, int64_t dim, int64_t num_entries,
    float scale, FastDiv by_nvec) {
  constexpr int V = emb_vec<WT, OT>();
  using index_t = std::conditional_t<BIG, int64_t, uint32_t>;
  index_t const total = (index_t)(num_bags * nvec);
  index_t const stride = (index_t)gridDim.x * kEmbThreads;
  for (index_t i = (index_t)blockIdx.x * kEmbThreads + threadIdx.x; i < total; i += stride) {
    int64_t b;
    int v;
    if constexpr (BIG) {
      b = i / nvec;
      v = (int)(i % nvec);
    } else {
      uint32_t q, r;
      by_nvec.divmod(i, q, r);
      b = q;
      v = (int)r;
    }
    float acc[V];
#pragma unroll
    for (int e = 0; e < V; e++) acc[e] = 0.0f;
    IT const *ib = idx + b * bag;
    int j = 0;
    // Bags of eight entries and more: eight row reads in flight, and the indices of the next
    // eight are asked for before this group's rows are waited for, so a bag of 32 costs one
    // index round trip and four row round trips instead of eight of each.  The sum keeps the
    // order of the entries.
    if constexpr (CHUNKED) {
      constexpr int CH = 8;
      int64_t rn[CH];
#pragma unroll
      for (int u = 0; u < CH; u++) rn[u] = (int64_t)ib[u];
      for (; j + CH <= bag; j += CH) {
        float w[CH][V];
        bool ok[CH];
#pragma unroll
        for (int u = 0; u < CH; u++) {
          ok[u] = (uint64_t)rn[u] < (uint64_t)num_entries;
          load_row<WT, V>(W + (ok[u] ? rn[u] : 0) * dim + (int64_t)v * V, w[u]);
        }
        if (j + 2 * CH <= bag) {
#pragma unroll
          for (int u = 0; u < CH; u++) rn[u] = (int64_t)ib[j + CH + u];
        }
#pragma unroll
        for (int u = 0; u < CH; u++)
#pragma unroll
          for (int e = 0; e < V; e++) acc[e] = acc[e] + (ok[u] ? w[u][e] : 0.0f);
      }
    }
    for (; j + 4 <= bag; j += 4) {  // four row reads in flight
      int64_t r[4];
      float w[4][V];
#pragma unroll
      for (int u = 0; u < 4; u++) r[u] = (int64_t)ib[j + u];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        bool ok = (uint64_t)r[u] < (uint64_t)num_entries;
        load_row<WT, V>(W + (ok ? r[u] : 0) * dim + (int64_t)v * V, w[u]);
        if (!ok) {
#pragma unroll
          for (int e = 0; e < V; e++) w[u][e] = 0.0f;
        }
      }
#pragma unroll
      for (int u = 0; u < 4; u++)
#pragma unroll
        for (int e = 0; e < V; e++) acc[e] = acc[e] + w[u][e];
    }
    for (; j < bag; j++) {
      int64_t r = (int64_t)ib[j];
      if ((uint64_t)r < (uint64_t)num_entries) {
        float w[V];
        load_row<WT, V>(W + r * dim + (int64_t)v * V, w);
#pragma unroll
        for (int e = 0; e < V; e++) acc[e] = acc[e] + w[e];
      }
    }
    if (scale != 1.0f) {
#pragma unroll
      for (int e = 0; e < V; e++) acc[e] *= scale;
    }
    store_out<OT, V>(out + b * dim + (int64_t)v * V, acc);
  }
}

template <typename IT, typename WT, typename OT>
__global__ __launch_bounds__(kEmbThreads) void embedding_fwd_scalar_kernel(
    IT const *__restrict__ idx, OT *__restrict__ out, WT const *__restrict__ W,
    int64_t num_bags, int bag, int64_t dim, int64_t num_entries, float scale) {
  int64_t const total = num_bags * dim;
  int64_t const stride = (int64_t)gridDim.x * kEmbThreads;
  for (int64_t i = (int64_t)blockIdx.x * kEmbThreads + threadIdx.x; i < total; i += stride) {
    int64_t const b = i / dim, d = i % dim;
    float acc = 0.0f;
    for (int j = 0; j < bag; j++) {
      int64_t r = (int64_t)idx[b * bag + j];
      if ((uint64_t)r < (uint64_t)num_entries) {
        acc = acc + VecIO<WT>::load1(W + r * dim + d);
      }
    }
    if (scale != 1.0f) acc *= scale;
    VecIO<OT>::store1(out + b * dim + d, acc);
  }
}

// HALF and DOUBLE tables (embedding_kernels.cu:374-449,491-566 forward, 609-808 backward): table,
// output and gradients share one type T and all arithmetic is T's own, as in the reference -- a bag
// is summed in T entry by entry, the backward adds T values atomically.  One thread per (bag,
// column); no configuration uses these types, so nothing here is tuned.
template <typename IT, typename T>
__global__ __launch_bounds__(kEmbThreads) void embedding_fwd_typed_kernel(
    IT const *__restrict__ idx, T *__restrict__ out, T const *__restrict__ W,
    int64_t num_bags, int bag, int64_t dim, int64_t num_entries, bool avg) {
  int64_t const total = num_bags * dim;
  int64_t const stride = (int64_t)gridDim.x * kEmbThreads;
  T const scale = (T)(1.0f / (float)bag);  // the reference's `TD scale = 1.0f / in_dim`
  for (int64_t i = (int64_t)blockIdx.x * kEmbThreads + threadIdx.x; i < total; i += stride) {
    int64_t const b = i / dim, d = i % dim;
    T acc = (T)0;
    for (int j = 0; j < bag; j++) {
      int64_t const r = (int64_t)idx[b * bag + j];
      if ((uint64_t)r < (uint64_t)num_entries) acc = acc + W[r * dim + d];
    }
    if (avg) acc = acc * scale;
    out[i] = acc;
  }
}

__device__ __forceinline__ void atomic_add_typed(double *p, double v) { atomicAdd(p, v); }
// no 16-bit atomic: compare-and-swap on the aligned word that holds the half
__device__ __forceinline__ void atomic_add_typed(_Float16 *p, _Float16 v) {
  uintptr_t const a = reinterpret_cast<uintptr_t>(p);
  uint32_t *word = reinterpret_cast<uint32_t *>(a & ~(uintptr_t)3);
  bool const high = (a & 2) != 0;
  uint32_t seen = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  for (;;) {
    uint16_t const bits = high ? (uint16_t)(seen >> 16) : (uint16_t)(seen & 0xffffu);
    _Float16 const sum = __builtin_bit_cast(_Float16, bits) + v;
    uint32_t const sb = __builtin_bit_cast(uint16_t, sum);
    uint32_t const want = high ? (seen & 0x0000ffffu) | (sb << 16) : (seen & 0xffff0000u) | sb;
    uint32_t const prev = atomicCAS(word, seen, want);
    if (prev == seen) break;
    seen = prev;
  }
}

template <typename IT, typename T>
__global__ __launch_bounds__(kEmbThreads) void embedding_bwd_typed_kernel(
    IT const *__restrict__ idx, T const *__restrict__ dY, T *dW,
    int64_t num_bags, int bag, int64_t dim, int64_t num_entries, bool avg) {
  int64_t const total = num_bags * dim;
  int64_t const stride = (int64_t)gridDim.x * kEmbThreads;
  T const scale = (T)(1.0f / (float)bag);
  for (int64_t i = (int64_t)blockIdx.x * kEmbThreads + threadIdx.x; i < total; i += stride) {
    int64_t const b = i / dim, d = i % dim;
    T g = dY[i];
    if (avg) g = g * scale;
    for (int j = 0; j < bag; j++) {
      int64_t const r = (int64_t)idx[b * bag + j];
      if ((uint64_t)r < (uint64_t)num_entries) atomic_add_typed(dW + r * dim + d, g);
    }
  }
}

// One wave per (bag, 64-float column segment): every atomic instruction of the
// wave covers 256 contiguous bytes of one weight-gradient row.
template <typename IT, typename GT>
__global__ __launch_bounds__(kEmbThreads) void embedding_bwd_atomic_kernel(
    IT const *__restrict__ idx, GT const *__restrict__ dY, float *dW,
    int64_t num_bags, int bag, int64_t dim, int64_t num_entries, float scale) {
  int const lane = threadIdx.x & 63;
  int64_t const segs = ceil_div(dim, 64);
  int64_t const total = num_bags * segs;
  int64_t const wave0 = ((int64_t)blockIdx.x * kEmbThreads + threadIdx.x) >> 6;
  int64_t const nwaves = ((int64_t)gridDim.x * kEmbThreads) >> 6;
  for (int64_t w = wave0; w < total; w += nwaves) {
    int64_t const b = w / segs;
    int64_t const d = (w % segs) * 64 + lane;
    if (d < dim) {
      float g = VecIO<GT>::load1(dY + b * dim + d);
      if (scale != 1.0f) g *= scale;
      for (int j = 0; j < bag; j++) {
        int64_t r = (int64_t)idx[b * bag + j];
        if ((uint64_t)r < (uint64_t)num_entries) {
          atomicAdd(dW + r * dim + d, g);
        }
      }
    }
  }
}

// Sorted scatter-add.  The atomic kernel above is bound by the rate at which
// the memory side retires fp32 atomics (about 0.7 TB/s of payload measured on
// MI355X, far below HBM).  With scratch from the caller the lookups are sorted
// by row id first (the stable radix sort of radix_sort.h); equal ids then
// form runs, a walker sums the gradient rows of a run in registers and adds the
// sum to the weight-gradient row with ordinary loads and stores, because a run
// that lies inside one walker's chunk is touched by nobody else.  Only runs
// that cross a chunk border (at most two per walker) go through atomics.
constexpr int kEmbChunk = 16;  // sorted positions per walker

// STREAM: the row is read once (one lookup per gradient row), so it need not stay in the caches.
template <typename V, bool STREAM>
__device__ __forceinline__ V load_grad_vec(void const *p) {
  if constexpr (STREAM) return __builtin_nontemporal_load(reinterpret_cast<V const *>(p));
  else return *reinterpret_cast<V const *>(p);
}
template <bool STREAM>
__device__ __forceinline__ void load_grad4(float const *p, float (&v)[4]) {
  f32x4 r = load_grad_vec<f32x4, STREAM>(p);
  v[0] = r[0]; v[1] = r[1]; v[2] = r[2]; v[3] = r[3];
}
template <bool STREAM>
__device__ __forceinline__ void load_grad4(bf16 const *p, float (&v)[4]) {
  u32x2 r = load_grad_vec<u32x2, STREAM>(p);
  v[0] = __uint_as_float(r[0] << 16);
  v[1] = __uint_as_float(r[0] & 0xffff0000u);
  v[2] = __uint_as_float(r[1] << 16);
  v[3] = __uint_as_float(r[1] & 0xffff0000u);
}

// LPR lanes share a row, 4 columns per lane and CPL such chunks per lane in
// one pass (columns c = ((k * LPR) + lane) * 4, k < CPL).
// A walker owns every run that STARTS in its chunk and follows it to its
// end, however far; no run is shared, nothing is atomic, and every row is
// summed in ascending lookup order, so the result is bit-reproducible (a very
// popular row is then summed by a single walker, which is slow).
template <typename GT, int LPR, int CPL>
__global__ __launch_bounds__(256) void embedding_bwd_sorted_kernel(
    uint32_t const *__restrict__ keys, uint32_t const *__restrict__ vals,
    GT const *__restrict__ dY, float *dW, int64_t n, int bag, int64_t dim,
    uint32_t invalid_key, float scale) {
  int64_t const walker = ((int64_t)blockIdx.x * 256 + threadIdx.x) / LPR;
  int const wl = threadIdx.x % LPR;
  int64_t const p0 = walker * kEmbChunk;
  if (p0 >= n) return;
  int64_t const p1 = min(p0 + (int64_t)kEmbChunk, n);
  int64_t start = p0;
  while (start < p1 && start > 0 && keys[start - 1] == keys[start]) start++;
  if (start >= p1) return;
  // is position p part of this walker's work?
  auto mine = [&](int64_t p) { return p < p1 || (p < n && keys[p] == keys[p - 1]); };
  for (int64_t cbase = 0; cbase < dim; cbase += (int64_t)LPR * 4 * CPL) {
    float acc[CPL][4], cur[CPL][4], nxt[CPL][4];
    auto fetch = [&](int64_t p, float (&v)[CPL][4]) {
      int64_t const l = (int64_t)vals[p];
      GT const *row = dY + (l / bag) * dim;
#pragma unroll
      for (int k = 0; k < CPL; k++) {
        int64_t const c = cbase + ((int64_t)k * LPR + wl) * 4;
        if (c < dim) {
          load_grad4<true>(row + c, v[k]);
        } else {
          v[k][0] = v[k][1] = v[k][2] = v[k][3] = 0.0f;
        }
      }
    };
#pragma unroll
    for (int k = 0; k < CPL; k++)
#pragma unroll
      for (int e = 0; e < 4; e++) acc[k][e] = 0.0f;
    fetch(start, cur);
    for (int64_t p = start; mine(p); p++) {
      bool const more = mine(p + 1);
      if (more) fetch(p + 1, nxt);  // next row in flight while this one is added
      uint32_t const id = keys[p];
#pragma unroll
      for (int k = 0; k < CPL; k++)
#pragma unroll
        for (int e = 0; e < 4; e++) acc[k][e] += cur[k][e];
      if (!more || keys[p + 1] != id) {  // the run's end
        if (id != invalid_key) {
#pragma unroll
          for (int k = 0; k < CPL; k++) {
            int64_t const c = cbase + ((int64_t)k * LPR + wl) * 4;
            if (c < dim) {
              float *dst = dW + (int64_t)id * dim + c;
              f32x4 old = *reinterpret_cast<f32x4 const *>(dst);
              f32x4 upd = {old[0] + acc[k][0] * scale, old[1] + acc[k][1] * scale,
                           old[2] + acc[k][2] * scale, old[3] + acc[k][3] * scale};
              *reinterpret_cast<f32x4 *>(dst) = upd;
            }
          }
        }
#pragma unroll
        for (int k = 0; k < CPL; k++)
#pragma unroll
          for (int e = 0; e < 4; e++) acc[k][e] = 0.0f;
      }
#pragma unroll
      for (int k = 0; k < CPL; k++)
#pragma unroll
        for (int e = 0; e < 4; e++) cur[k][e] = nxt[k][e];
    }
  }
}

// The non-deterministic sorted path of bags between two ends (the rule in emb_backward) and of tensors of 4 GB and
// more, which the walk's 32-bit offsets (embedding_walk.h) do not reach: a wave walks `chunk` consecutive sorted positions, a
// workgroup sixteen such chunks.  Walkers add runs that lie inside their chunk straight to memory;
// the partial sums of runs that cross a walker border meet in LDS and are merged by the workgroup,
// so only runs that cross a WORKGROUP border reach memory as atomics.  A row looked up
// thousands of times (Zipf-distributed tokens) then costs one atomic per
// element per workgroup instead of one per walker, which matters because
// atomics to one address are retired one after the other.
// A walker is a whole wave whatever the row length (VPL columns per lane; blockIdx.y takes the next
// 256 columns of longer rows): ids, row addresses and the run logic are then scalar work beside the loads.  With two
// walkers to a wave (dim 128) every position took about a hundred vector instructions, and
// they, not memory, were the bound (524 288 lookups in bags of 32, 1 M rows of 128
// floats: 78 -> 56 us; 65 536 lookups of 1024 bf16 columns, which had a wave to a walker before: 64 -> 58).
constexpr int kEmbBlockThreads = 1024;
constexpr int kEmbWalkers = kEmbBlockThreads / 64;
constexpr int kEmbMaxChunk = 64;  // one (row id, lookup) pair per lane

template <int VPL, bool STREAM>
__device__ __forceinline__ void load_grad_piece(float const *p, float (&v)[VPL]) {
  using vec = typename std::conditional<VPL == 4, f32x4, typename std::conditional<VPL == 2, f32x2, float>::type>::type;
  vec const r = load_grad_vec<vec, STREAM>(p);
  if constexpr (VPL == 1) {
    v[0] = r;
  } else {
#pragma unroll
    for (int e = 0; e < VPL; e++) v[e] = r[e];
  }
}
template <int VPL, bool STREAM>
__device__ __forceinline__ void load_grad_piece(bf16 const *p, float (&v)[VPL]) {
  using word = typename std::conditional<VPL == 4, u32x2, typename std::conditional<VPL == 2, uint32_t, uint16_t>::type>::type;
  word const r = load_grad_vec<word, STREAM>(p);
  if constexpr (VPL == 1) {
    v[0] = __uint_as_float((uint32_t)r << 16);
  } else if constexpr (VPL == 2) {
    v[0] = __uint_as_float(r << 16);
    v[1] = __uint_as_float(r & 0xffff0000u);
  } else {
    v[0] = __uint_as_float(r[0] << 16);
    v[1] = __uint_as_float(r[0] & 0xffff0000u);
    v[2] = __uint_as_float(r[1] << 16);
    v[3] = __uint_as_float(r[1] & 0xffff0000u);
  }
}

// DEPTH positions in flight, as many as fit the registers that let two workgroups share a CU.
// BAGGED: bags of several entries, whose gradient row the walkers read once per entry: cached loads.
template <typename GT, int VPL, bool BAGGED>
__global__ __launch_bounds__(kEmbBlockThreads, 8) void embedding_bwd_sorted_block_kernel(
    uint32_t const *__restrict__ keys, uint32_t const *__restrict__ vals,
    GT const *__restrict__ dY, float *dW, int64_t n, int chunk, int bag, int dim,
    uint32_t invalid_key, float scale) {
  constexpr int PW = 64 * VPL;  // columns of a workgroup
  constexpr int DEPTH = VPL == 4 ? 4 : 8;
  __shared__ float emb_part[2 * kEmbWalkers * PW];  // border partials
  __shared__ uint32_t part_id[2 * kEmbWalkers];
  __shared__ int part_valid[2 * kEmbWalkers];
  int const lane = threadIdx.x & 63;
  int const w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int64_t const block0 = (int64_t)blockIdx.x * kEmbWalkers * chunk;
  int64_t const block1 = min(block0 + (int64_t)kEmbWalkers * chunk, n);
  int64_t const p0 = block0 + (int64_t)w * chunk;
  int64_t const p1 = min(p0 + (int64_t)chunk, n);
  // The walker's (row id, lookup) pairs are fetched once, one pair per lane, and read back as
  // scalars.  What the walk would otherwise wait for at every position -- the gradient row of the
  // lookup and, where a run ends, the weight-gradient row it is added to -- is then asked for
  // DEPTH positions ahead.
  int const cnt = (int)max((int64_t)0, min((int64_t)chunk, n - p0));  // positions that exist
  uint32_t my_key = invalid_key, my_val = 0;
  if (lane < cnt) {
    my_key = keys[p0 + lane];
    my_val = vals[p0 + lane];
    // what the walk needs of a lookup is the gradient row it reads: its bag
    if (BAGGED) my_val /= (uint32_t)bag;
  }
  uint32_t const key_before = cnt > 0 && p0 > 0 ? keys[p0 - 1] : invalid_key;
  uint32_t const key_after = cnt > 0 && p1 < n ? keys[p1] : invalid_key;
  auto key_at = [&](int j) { return (uint32_t)__builtin_amdgcn_readlane((int)my_key, j); };  // j < cnt
  auto next_key = [&](int j) { return j + 1 < cnt ? key_at(j + 1) : key_after; };
  bool const head_shared = cnt > 0 && p0 > 0 && key_before == key_at(0);

  // this lane's columns, and those it reads instead where the row ends before them
  uint32_t const col = blockIdx.y * PW + lane * VPL;
  uint32_t const safe = col < (uint32_t)dim ? col : blockIdx.y * PW;
  auto store_piece = [&](float *row, float const (&v)[VPL]) {
    if (col >= (uint32_t)dim) return;
    if constexpr (VPL == 4) *reinterpret_cast<f32x4 *>(row + col) = f32x4{v[0], v[1], v[2], v[3]};
    else if constexpr (VPL == 2) *reinterpret_cast<f32x2 *>(row + col) = f32x2{v[0], v[1]};
    else row[col] = v[0];
  };
  if (lane == 0) {
    part_valid[2 * w] = 0;
    part_valid[2 * w + 1] = 0;
  }
  {
    float acc[VPL], rows[DEPTH][VPL], old[DEPTH][VPL];
    // position j's gradient row, and the weight-gradient row of its id if a run of this
    // walker alone ends there (nobody else touches that row during the kernel)
    auto prefetch = [&](int j, float (&v)[VPL], float (&o)[VPL]) {
      if (j >= cnt) return;
      uint32_t const id = key_at(j);
      GT const *row = dY + (int64_t)(uint32_t)__builtin_amdgcn_readlane((int)my_val, j) * dim;
      load_grad_piece<VPL, !BAGGED>(row + safe, v);
      if (next_key(j) != id && id != invalid_key) {
        float const *dst = dW + (int64_t)id * dim;
        load_grad_piece<VPL, false>(dst + safe, o);
      }
    };
    bool shared_run = head_shared;
    auto step = [&](int j, float (&v)[VPL], float (&o)[VPL]) {
      if (j >= cnt) return;
      uint32_t const id = key_at(j);
#pragma unroll
      for (int e = 0; e < VPL; e++) acc[e] += v[e];
      bool const tail_shared = j + 1 == cnt && p1 < n && key_after == id;
      if (tail_shared || j + 1 == cnt || next_key(j) != id) {
        if (id != invalid_key) {
          if (shared_run || tail_shared) {
            // slot 2w: run shared with the previous walker (or both sides);
            // slot 2w+1: run shared with the next walker only
            int const slot = shared_run ? 2 * w : 2 * w + 1;
#pragma unroll
            for (int e = 0; e < VPL; e++) emb_part[slot * PW + e * 64 + lane] = acc[e];
            if (lane == 0) {
              part_id[slot] = id;
              // 1: a border partial; 2 / 4: its run also extends before /
              // beyond the workgroup's positions
              part_valid[slot] = 1 | ((shared_run && p0 == block0) ? 2 : 0) |
                                 ((tail_shared && p1 == block1) ? 4 : 0);
            }
          } else {
            float *dst = dW + (int64_t)id * dim;
            float u[VPL];
#pragma unroll
            for (int e = 0; e < VPL; e++) u[e] = o[e] + acc[e] * scale;
            store_piece(dst, u);
          }
        }
        shared_run = false;
#pragma unroll
        for (int e = 0; e < VPL; e++) acc[e] = 0.0f;
      }
      // this slot is free now: position j + DEPTH goes into it
      prefetch(j + DEPTH, v, o);
    };
#pragma unroll
    for (int e = 0; e < VPL; e++) acc[e] = 0.0f;
#pragma unroll
    for (int j = 0; j < DEPTH; j++) prefetch(j, rows[j], old[j]);
#pragma unroll 1
    for (int j = 0; j < cnt; j += DEPTH) {
#pragma unroll
      for (int u = 0; u < DEPTH; u++) step(j + u, rows[u], old[u]);
    }
  }
  __syncthreads();
  // Merge the border partials.  A run that crosses walkers has one partial per walker: the one
  // it starts in (slot 2w+1, or slot 0 if it comes from the workgroup before) and slot 2w of
  // each walker it reaches.  The walker of the first adds them up in position order, all runs
  // side by side.
  for (int sidx = w == 0 ? 0 : 2 * w + 1; sidx <= 2 * w + 1; sidx++) {
    int flags = __builtin_amdgcn_readfirstlane(part_valid[sidx]);
    if (flags == 0) continue;
    uint32_t const id = (uint32_t)__builtin_amdgcn_readfirstlane((int)part_id[sidx]);
    float acc[VPL];
#pragma unroll
    for (int e = 0; e < VPL; e++) acc[e] = emb_part[sidx * PW + e * 64 + lane];
    for (int nxt = (sidx | 1) + 1; nxt < 2 * kEmbWalkers && part_valid[nxt] != 0 && part_id[nxt] == id; nxt += 2) {
      flags |= part_valid[nxt];
#pragma unroll
      for (int e = 0; e < VPL; e++) acc[e] += emb_part[nxt * PW + e * 64 + lane];
    }
    float *dst = dW + (int64_t)id * dim;
    if ((flags & 6) != 0) {
      if (col < (uint32_t)dim) {
#pragma unroll
        for (int e = 0; e < VPL; e++) atomicAdd(dst + col + e, acc[e] * scale);
      }
    } else {
      float u[VPL];
      load_grad_piece<VPL, false>(dst + safe, u);
#pragma unroll
      for (int e = 0; e < VPL; e++) u[e] += acc[e] * scale;
      store_piece(dst, u);
    }
  }
}

// Scratch layout: keys A | keys B | lookups A | lookups B | digit table of the sort
struct EmbSortLayout {
  size_t keys_a, keys_b, vals_a, vals_b, table, total;
  RadixSortPlan plan;
};

static unsigned key_bits(int64_t num_entries) {
  unsigned b = 1;
  while (b < 32 && ((int64_t)1 << b) <= num_entries) b++;
  return b;
}

static bool emb_sort_layout(int64_t n, int64_t num_entries, EmbSortLayout &L) {
  if (n <= 0 || n >= (1ll << 31) || num_entries >= 0xffffffffll) return false;
  L.plan = radix_sort_plan(n, key_bits(num_entries));
  size_t const arr = ((size_t)n * 4 + 255) & ~(size_t)255;
  L.keys_a = 0;
  L.keys_b = arr;
  L.vals_a = 2 * arr;
  L.vals_b = 3 * arr;
  L.table = 4 * arr;
  L.total = 4 * arr + ((L.plan.table_bytes + 255) & ~(size_t)255);
  return true;
}

static int emb_grid(int64_t threads_needed) {
  int64_t b = ceil_div(threads_needed > 0 ? threads_needed : 1, kEmbThreads);
  int64_t const cap = (int64_t)kNumCU * 256;
  return (int)(b < cap ? b : cap);
}

template <typename IT, typename WT, typename OT>
static int emb_forward(hipStream_t st, void const *indices, void *output,
                       void const *weight, int64_t num_bags, int64_t bag,
                       int64_t dim, int64_t num_entries, float scale) {
  constexpr int V = emb_vec<WT, OT>();
  IT const *I = static_cast<IT const *>(indices);
  WT const *W = static_cast<WT const *>(weight);
  OT *O = static_cast<OT *>(output);
  if (dim % V == 0 && aligned16(weight) && aligned16(output)) {
    int nvec = (int)(dim / V);
    // 32-bit thread indices while index + one grid stride cannot wrap
    bool const fast = num_bags * nvec < ((int64_t)1 << 31) - (int64_t)kNumCU * 256 * kEmbThreads;
    FastDiv const by_nvec = fast ? make_fast_div((uint32_t)nvec) : FastDiv{};
#define FFK_EMB_FWD(BIG_, CHUNKED_)                                                                   \
  embedding_fwd_vec_kernel<IT, WT, OT, BIG_, CHUNKED_><<<emb_grid(num_bags * nvec), kEmbThreads, 0, st>>>( \
      I, O, W, num_bags, (int)bag, nvec, dim, num_entries, scale, by_nvec)
    if (bag >= 8) {
      if (fast) FFK_EMB_FWD(false, true);
      else FFK_EMB_FWD(true, true);
    } else {
      if (fast) FFK_EMB_FWD(false, false);
      else FFK_EMB_FWD(true, false);
    }
#undef FFK_EMB_FWD
  } else {
    embedding_fwd_scalar_kernel<IT, WT, OT><<<emb_grid(num_bags * dim), kEmbThreads, 0, st>>>(
        I, O, W, num_bags, (int)bag, dim, num_entries, scale);
  }
  FFK_CHECK_LAUNCH();
  return FFK_OK;
}

template <typename IT, typename GT>
static int emb_backward(hipStream_t st, void const *indices, void const *dy,
                        float *dw, int64_t num_bags, int64_t bag, int64_t dim,
                        int64_t num_entries, float scale, void *workspace,
                        size_t workspace_bytes, bool deterministic) {
  int64_t const lookups = num_bags * bag;
  // A caller without the scratch gets atomics whatever the sizes: calls on several streams may then add to one
  // table at a time.  The kernels behind the scratch add to a row with loads and stores.
  EmbSortLayout L;
  bool const alone = workspace != nullptr && reinterpret_cast<uintptr_t>(workspace) % 256 == 0 &&
                     emb_sort_layout(lookups, num_entries, L) && L.total <= workspace_bytes;
  bool const vectors = dim % 4 == 0 && aligned16(dy) && aligned16(dw);
  if (alone && vectors && !deterministic && embedding_match_takes(lookups, dim, num_entries)) {
    FFK_HIP(embedding_match<IT>(st, static_cast<IT const *>(indices), static_cast<GT const *>(dy), dw, (int)lookups, (int)bag,
                                (int)dim, num_entries, scale));
    return FFK_OK;
  }
  bool const sorted = alone && vectors && (deterministic || dim <= 65535 * 256);  // the walk's grid takes 256 columns a row
  if (sorted) {
    uint8_t *ws = static_cast<uint8_t *>(workspace);
    uint32_t *keys_out = nullptr, *vals_out = nullptr;
    FFK_HIP(radix_sort_lookups<IT>(st, static_cast<IT const *>(indices), lookups, num_entries, L.plan,
                                   reinterpret_cast<uint32_t *>(ws + L.keys_a), reinterpret_cast<uint32_t *>(ws + L.keys_b),
                                   reinterpret_cast<uint32_t *>(ws + L.vals_a), reinterpret_cast<uint32_t *>(ws + L.vals_b),
                                   reinterpret_cast<uint32_t *>(ws + L.table), &keys_out, &vals_out));
    GT const *G = static_cast<GT const *>(dy);
    if (deterministic) {
      int64_t const walkers = ceil_div(lookups, kEmbChunk);
#define FFK_EMB_SORTED(LPR_, CPL_)                                             \
  embedding_bwd_sorted_kernel<GT, LPR_, CPL_><<<(unsigned)ceil_div(walkers * LPR_, 256), 256, 0, st>>>( \
      keys_out, vals_out, G, dw, lookups, (int)bag, dim, (uint32_t)num_entries, scale)
      if (dim > 512) FFK_EMB_SORTED(64, 4);
      else if (dim > 256) FFK_EMB_SORTED(64, 2);
      else if (dim > 128) FFK_EMB_SORTED(64, 1);
      else if (dim > 64) FFK_EMB_SORTED(32, 1);
      else FFK_EMB_SORTED(16, 1);
#undef FFK_EMB_SORTED
      FFK_CHECK_LAUNCH();
      return FFK_OK;
    }
    // 32-bit byte offsets reach all of both tensors.  Not bags of 65 to 128 columns with 65 536 lookups and
    // up to four times as many, where the kernel below is ahead (a table's pass, us, that kernel and the walk; 128 columns:
    // 40 000 lookups 38.0 37.6, 85 700 49.2 52.0, 138 264 58.5 66.3, 200 000 70.9 76.5, 300 000 of 900 000 rows 93.8 90.5,
    // 524 288 127 116; 96 columns: 138 264 56.5 61.8, 300 000 80.2 76.3; 64 columns: 54.6 56.0 of 50 000 rows, 61.3 58.0 of
    // 900 000).
    bool const middling = bag > 1 && dim > 64 && dim <= 128 && lookups >= (1 << 16) && lookups < (1 << 18);
    if (!middling && (uint64_t)num_entries * dim * 4 <= kWalkNowhere && (uint64_t)num_bags * dim * sizeof(GT) <= kWalkNowhere) {
      WalkArgs const a = {keys_out, vals_out, lookups, 0, (int)bag, (int)dim, (uint32_t)num_entries, scale,
                          (uint32_t)(num_bags * dim * (int64_t)sizeof(GT)), (uint32_t)(num_entries * dim * 4)};
      FFK_HIP(embedding_walk<GT>(st, a, G, dw));
      return FFK_OK;
    }
    // Longer chunks mean fewer border partials and fewer atomics on hot rows; 8192 walkers are every
    // wave the chip holds (sort and walk of 524 288 x 128: 96.8 us, 99 with 16384 walkers, 109 with 32768;
    // of 65 536 x 1024 bf16: 77, 81.6, 81.5).
    int64_t const groups = ceil_div(dim, 256);
    int const chunk =
        (int)std::min<int64_t>(kEmbMaxChunk, std::max<int64_t>(kEmbChunk, ceil_div(lookups * groups, 8192)));
    dim3 const blocks((unsigned)ceil_div(lookups, (int64_t)kEmbWalkers * chunk), (unsigned)groups);
#define FFK_EMB_SORTED(VPL_)                                                   \
  do {                                                                         \
    auto kern = bag > 1 ? embedding_bwd_sorted_block_kernel<GT, VPL_, true>    \
                        : embedding_bwd_sorted_block_kernel<GT, VPL_, false>;  \
    kern<<<blocks, kEmbBlockThreads, 0, st>>>(keys_out, vals_out, G, dw, lookups, chunk, (int)bag, (int)dim, \
                                              (uint32_t)num_entries, scale);   \
  } while (0)
    if (dim > 128) FFK_EMB_SORTED(4);
    else if (dim > 64) FFK_EMB_SORTED(2);
    else FFK_EMB_SORTED(1);
#undef FFK_EMB_SORTED
    FFK_CHECK_LAUNCH();
    return FFK_OK;
  }
  if (deterministic) {
    return fail(FFK_ERR_WORKSPACE,
                "embedding_backward: deterministic mode needs the sort workspace "
                "(ffk_embedding_backward_workspace_bytes), 256-byte aligned, and dim %% 4 == 0");
  }
  int64_t waves = num_bags * ceil_div(dim, 64);
  embedding_bwd_atomic_kernel<IT, GT><<<emb_grid(waves * 64), kEmbThreads, 0, st>>>(
      static_cast<IT const *>(indices), static_cast<GT const *>(dy), dw, num_bags,
      (int)bag, dim, num_entries, scale);
  FFK_CHECK_LAUNCH();
  return FFK_OK;
}

static int check_common(char const *who, int aggr, int64_t num_bags, int64_t bag,
                        int64_t dim, int64_t num_entries) {
  FFK_REQUIRE(num_bags >= 0 && bag > 0 && dim > 0 && num_entries > 0, "%s: bad shape", who);
  FFK_REQUIRE(bag < (1ll << 31), "%s: bag too large", who);
  FFK_REQUIRE(aggr >= FFK_AGGR_NONE && aggr <= FFK_AGGR_AVG, "%s: bad aggregate op %d", who, aggr);
  FFK_REQUIRE(aggr != FFK_AGGR_NONE || bag == 1, "%s: bag must be 1 without an aggregate op", who);
  return FFK_OK;
}

}  // namespace ffk

using namespace ffk;

extern "C" int ffk_embedding_forward(ffk_stream_t stream, int index_dtype,
                                     int weight_dtype, int output_dtype,
                                     void const *indices, void *output,
                                     void const *weight, int aggr,
                                     int64_t num_bags, int64_t bag, int64_t dim,
                                     int64_t num_entries) {
  int rc = check_common("embedding_forward", aggr, num_bags, bag, dim, num_entries);
  if (rc != FFK_OK) return rc;
  if (num_bags == 0) return FFK_OK;
  FFK_REQUIRE(indices && output && weight, "embedding_forward: NULL tensor");
  float scale = aggr == FFK_AGGR_AVG ? 1.0f / (float)bag : 1.0f;
  hipStream_t st = as_stream(stream);
#define FFK_EMB_FWD(IT, WT, OT)                                                \
  return emb_forward<IT, WT, OT>(st, indices, output, weight, num_bags, bag, dim, num_entries, scale)
  if (index_dtype == FFK_INT32) {
    if (weight_dtype == FFK_FLOAT && output_dtype == FFK_FLOAT) FFK_EMB_FWD(int32_t, float, float);
    if (weight_dtype == FFK_FLOAT && output_dtype == FFK_BF16) FFK_EMB_FWD(int32_t, float, bf16);
    if (weight_dtype == FFK_BF16 && output_dtype == FFK_BF16) FFK_EMB_FWD(int32_t, bf16, bf16);
    if (weight_dtype == FFK_BF16 && output_dtype == FFK_FLOAT) FFK_EMB_FWD(int32_t, bf16, float);
  } else if (index_dtype == FFK_INT64) {
    if (weight_dtype == FFK_FLOAT && output_dtype == FFK_FLOAT) FFK_EMB_FWD(int64_t, float, float);
    if (weight_dtype == FFK_FLOAT && output_dtype == FFK_BF16) FFK_EMB_FWD(int64_t, float, bf16);
    if (weight_dtype == FFK_BF16 && output_dtype == FFK_BF16) FFK_EMB_FWD(int64_t, bf16, bf16);
    if (weight_dtype == FFK_BF16 && output_dtype == FFK_FLOAT) FFK_EMB_FWD(int64_t, bf16, float);
  }
#undef FFK_EMB_FWD
  if (weight_dtype == output_dtype && (weight_dtype == FFK_HALF || weight_dtype == FFK_DOUBLE) &&
      (index_dtype == FFK_INT32 || index_dtype == FFK_INT64)) {
    bool const avg = aggr == FFK_AGGR_AVG;
    int const grid = emb_grid(num_bags * dim);
#define FFK_EMB_TYPED(IT, T)                                                   \
  embedding_fwd_typed_kernel<IT, T><<<grid, kEmbThreads, 0, st>>>(             \
      static_cast<IT const *>(indices), static_cast<T *>(output), static_cast<T const *>(weight), num_bags, (int)bag, \
      dim, num_entries, avg)
    if (index_dtype == FFK_INT32 && weight_dtype == FFK_HALF) FFK_EMB_TYPED(int32_t, _Float16);
    else if (index_dtype == FFK_INT32) FFK_EMB_TYPED(int32_t, double);
    else if (weight_dtype == FFK_HALF) FFK_EMB_TYPED(int64_t, _Float16);
    else FFK_EMB_TYPED(int64_t, double);
#undef FFK_EMB_TYPED
    FFK_CHECK_LAUNCH();
    return FFK_OK;
  }
  return fail(FFK_ERR_UNSUPPORTED,
              "embedding_forward: dtypes (index %d, weight %d, output %d) not supported",
              index_dtype, weight_dtype, output_dtype);
}

extern "C" size_t ffk_embedding_backward_workspace_bytes(int64_t num_indices,
                                                         int64_t num_entries) {
  EmbSortLayout L;
  if (!emb_sort_layout(num_indices, num_entries, L)) return 0;
  return L.total;
}

extern "C" int ffk_embedding_backward(ffk_stream_t stream, int index_dtype,
                                      int output_grad_dtype,
                                      void const *indices,
                                      void const *output_grad,
                                      float *weight_grad, int aggr,
                                      int64_t num_bags, int64_t bag,
                                      int64_t dim, int64_t num_entries,
                                      int deterministic, void *workspace,
                                      size_t workspace_bytes) {
  int rc = check_common("embedding_backward", aggr, num_bags, bag, dim, num_entries);
  if (rc != FFK_OK) return rc;
  if (num_bags == 0) return FFK_OK;
  FFK_REQUIRE(indices && output_grad && weight_grad, "embedding_backward: NULL tensor");
  float scale = aggr == FFK_AGGR_AVG ? 1.0f / (float)bag : 1.0f;
  hipStream_t st = as_stream(stream);
#define FFK_EMB_BWD(IT, GT)                                                    \
  return emb_backward<IT, GT>(st, indices, output_grad, weight_grad, num_bags, bag, dim, num_entries, scale, \
                              workspace, workspace_bytes, deterministic != 0)
  if (index_dtype == FFK_INT32) {
    if (output_grad_dtype == FFK_FLOAT) FFK_EMB_BWD(int32_t, float);
    if (output_grad_dtype == FFK_BF16) FFK_EMB_BWD(int32_t, bf16);
  } else if (index_dtype == FFK_INT64) {
    if (output_grad_dtype == FFK_FLOAT) FFK_EMB_BWD(int64_t, float);
    if (output_grad_dtype == FFK_BF16) FFK_EMB_BWD(int64_t, bf16);
  }
#undef FFK_EMB_BWD
  return fail(FFK_ERR_UNSUPPORTED,
              "embedding_backward: dtypes (index %d, grad %d) not supported",
              index_dtype, output_grad_dtype);
}

extern "C" int ffk_embedding_backward_typed(ffk_stream_t stream, int index_dtype, int dtype,
                                            void const *indices, void const *output_grad,
                                            void *weight_grad, int aggr, int64_t num_bags,
                                            int64_t bag, int64_t dim, int64_t num_entries) {
  if (dtype == FFK_FLOAT) {
    return ffk_embedding_backward(stream, index_dtype, FFK_FLOAT, indices, output_grad,
                                  static_cast<float *>(weight_grad), aggr, num_bags, bag, dim, num_entries, 0,
                                  nullptr, 0);
  }
  int rc = check_common("embedding_backward_typed", aggr, num_bags, bag, dim, num_entries);
  if (rc != FFK_OK) return rc;
  FFK_REQUIRE(dtype == FFK_HALF || dtype == FFK_DOUBLE,
              "embedding_backward_typed: dtype %d not supported (HALF, FLOAT or DOUBLE)", dtype);
  FFK_REQUIRE(index_dtype == FFK_INT32 || index_dtype == FFK_INT64,
              "embedding_backward_typed: index dtype %d not supported", index_dtype);
  if (num_bags == 0) return FFK_OK;
  FFK_REQUIRE(indices && output_grad && weight_grad, "embedding_backward_typed: NULL tensor");
  hipStream_t st = as_stream(stream);
  bool const avg = aggr == FFK_AGGR_AVG;
  int const grid = emb_grid(num_bags * dim);
#define FFK_EMB_TYPED(IT, T)                                                   \
  embedding_bwd_typed_kernel<IT, T><<<grid, kEmbThreads, 0, st>>>(             \
      static_cast<IT const *>(indices), static_cast<T const *>(output_grad), static_cast<T *>(weight_grad), num_bags, \
      (int)bag, dim, num_entries, avg)
  if (index_dtype == FFK_INT32 && dtype == FFK_HALF) FFK_EMB_TYPED(int32_t, _Float16);
  else if (index_dtype == FFK_INT32) FFK_EMB_TYPED(int32_t, double);
  else if (dtype == FFK_HALF) FFK_EMB_TYPED(int64_t, _Float16);
  else FFK_EMB_TYPED(int64_t, double);
#undef FFK_EMB_TYPED
  FFK_CHECK_LAUNCH();
  return FFK_OK;
}
