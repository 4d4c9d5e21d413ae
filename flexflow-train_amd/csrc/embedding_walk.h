// The walk of a sorted scatter-add: positions of (row id, gradient row) in ascending row order, sums of
// equal ids added to the rows of the weight gradient.
//
// A walker is LPR lanes, four columns each, and takes `chunk` consecutive positions; a workgroup holds 16
// walkers of a whole wave (rows longer than 128, 256 columns at a time) or 32 narrower ones.  What a walker
// asks of a position is worked out beforehand, one position a thread, and laid into LDS: where its two rows
// lie and what becomes of the sum behind it.  A position then costs a wave one LDS read, the load of the
// gradient row, the load and the store of the weight-gradient row where a run ends, and some twenty vector
// instructions, for all its walkers at once.  (With a whole wave a walker and the run logic in scalar
// registers, read lane by lane, a position took the wave 300 cycles whether or not it touched memory: 524 288
// lookups in bags of 32, 128 floats a row, 57 us, 55 with all loads left out; 40 now where the weight gradient
// lies in the caches, 52 where it comes from memory.  14 us for the 6089 lookups of a small batch, 9 now.)
// An access past the end of the buffer, in the place of one that a position has no need of, costs a wave the
// 16 cycles of a 16-byte access all the same: branches around it are cheaper (50 us against 44).
// Workgroups go from the end of the positions to their beginning: where ids are ranked by how often they come
// up, the positions at the end are rows looked up once each, which take longest, and there are twice the
// walkers that the chip holds at a time, so that the others fill in behind them (65 536 x 1024 bf16
// with its sort, caches full of what another kernel wrote / read / of these tensors: 93 / 85 / 79 us in the order of the
// positions, 87 / 78 / 72 so; 55 139 x 328 bf16 50 / 46 / 43 and 53 / 49 / 44).
//
// Walkers add runs that lie inside their chunk straight to memory; the partial sums of runs that cross a
// walker border meet in LDS and are merged by the workgroup, so only runs that cross a WORKGROUP border
// reach memory as atomics: a row looked up thousands of times costs one atomic per element per workgroup.
#pragma once
#include "ffk_common.h"
#include <type_traits>

namespace ffk {

constexpr uint32_t kWalkNowhere = 0xfffff000u;  // a byte offset past every buffer, with a lane's columns added or not
constexpr int64_t kWalkWaves = 16384;  // twice what the chip holds

struct WalkArgs {
  uint32_t const *keys, *vals;  // sorted row ids, and the lookup each stands for
  int64_t n;
  int chunk_shift, bag, dim;
  uint32_t invalid_key;
  float scale;
  uint32_t dy_bytes, dw_bytes;  // of the two tensors
};

template <typename GT, int LPR>
struct WalkShape {
  static constexpr int kWalkers = LPR == 64 ? 16 : 32;
  static constexpr int kThreads = kWalkers * LPR;
  static constexpr int kMaxChunk = LPR >= 32 ? 64 : 16;  // positions of a walker
};

// BAGGED: bags of several entries, whose gradient rows are read once per entry; the weight gradient's then
// pass by the caches so that those stay (eight tables of 524 288 lookups 1056 us without that, 1036 with it).
// Otherwise a gradient row is read once, and passes by the caches: what it would drive out of them has to be written
// back first.  Sort and walk, us, with caches full of what another kernel wrote / read / of these tensors, and in
// brackets with gradient rows that go through the caches: 65 536 x 1024 bf16 82 / 76 / 70 (104 / 76 / 62), 16 384 x 1024
// bf16 43 / 39 / 34 (48 / 39 / 32), 55 139 x 328 bf16 48 / 46 / 42 (53 / 45 / 39), 21 193 x 1376 fp32 50 / 47 / 43 (72 /
// 48 / 40).
template <typename GT, int LPR, bool BAGGED>
__global__ __launch_bounds__((WalkShape<GT, LPR>::kThreads), (WalkShape<GT, LPR>::kThreads == 1024 ? 8 : 4))
void embedding_bwd_walk_kernel(WalkArgs a, GT const *dY, float *dW) {
  constexpr int WALKERS = WalkShape<GT, LPR>::kWalkers, NT = WalkShape<GT, LPR>::kThreads, PW = LPR * 4;
  constexpr int DEPTH = 4, kNonTemporal = 2;
  __shared__ u32x2 meta[WALKERS * WalkShape<GT, LPR>::kMaxChunk];
  __shared__ float emb_part[2 * WALKERS * PW];  // border partials
  __shared__ uint32_t part_id[2 * WALKERS];
  __shared__ int part_valid[2 * WALKERS];
  enum : uint32_t { kEnds = 1, kStore = 2, kPartial = 4, kHead = 8, kFlags = 15 };
  int const t = threadIdx.x, q = t / LPR, l = t % LPR;
  int const chunk = 1 << a.chunk_shift;
  int64_t const block0 = (int64_t)(gridDim.x - 1 - blockIdx.x) << (a.chunk_shift + (WALKERS == 16 ? 4 : 5));
  if (t < 2 * WALKERS) part_valid[t] = 0;
  __syncthreads();
  for (int i = t; i < WALKERS * chunk; i += NT) {
    int64_t const p = block0 + i, start = p & ~(int64_t)(chunk - 1);
    u32x2 m = {kWalkNowhere, 0u};
    if (p < a.n) {
      uint32_t const id = a.keys[p], val = a.vals[p];
      bool const more = p + 1 < a.n, last = p + 1 == start + chunk || !more;  // of the walker's positions
      uint32_t const next = more ? a.keys[p + 1] : 0u, before = start > 0 ? a.keys[start - 1] : 0u;
      bool const ends = last || next != id;
      // the run goes on behind the walker's positions, or began before them
      bool const tail = last && more && next == id, head = start > 0 && before == id;
      m[0] = (BAGGED ? val / (uint32_t)a.bag : val) * ((uint32_t)a.dim * (uint32_t)sizeof(GT));
      if (ends && id != a.invalid_key) {
        if (head || tail) {
          // slot 2w: run shared with the previous walker (or both sides);
          // slot 2w+1: run shared with the next walker only
          int const w = i >> a.chunk_shift, slot = head ? 2 * w : 2 * w + 1;
          part_id[slot] = id;
          // 1: a border partial; 2 / 4: its run also extends before /
          // beyond the workgroup's positions
          part_valid[slot] = 1 | (head && w == 0 ? 2 : 0) | (tail && w == WALKERS - 1 ? 4 : 0);
          m[1] = kPartial | (head ? kHead : 0u);
        } else {
          m[1] = id * ((uint32_t)a.dim * 4u) | kStore;
        }
      }
      m[1] |= ends ? kEnds : 0u;
    }
    meta[i] = m;
  }
  __syncthreads();
  uint32_t const col = blockIdx.y * PW + l * 4;  // this lane's first column
  if (col < (uint32_t)a.dim) {
    // buffers that begin at the workgroup's columns: kWalkNowhere and a lane's own columns do not wrap
    uint32_t const skip = blockIdx.y * PW, col_y = (uint32_t)l * 4u * (uint32_t)sizeof(GT), col_w = (uint32_t)l * 16u;
    __amdgpu_buffer_rsrc_t const ry =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<GT *>(dY) + skip, 0, (int)(a.dy_bytes - skip * (uint32_t)sizeof(GT)), 0x00020000);
    __amdgpu_buffer_rsrc_t const rw = __builtin_amdgcn_make_buffer_rsrc(dW + skip, 0, (int)(a.dw_bytes - skip * 4u), 0x00020000);
    u32x2 const *const mine = meta + (q << a.chunk_shift);
    using Raw = typename std::conditional<sizeof(GT) == 2, u32x2, u32x4>::type;
    constexpr int aux = BAGGED ? 0 : kNonTemporal;
    Raw rows[DEPTH];
    u32x4 old[DEPTH];
    uint32_t what[DEPTH];
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    auto prefetch = [&](int j, int u) __attribute__((always_inline)) {
      u32x2 m = mine[min(j, chunk - 1)];
      uint32_t const y = j < chunk ? m[0] : kWalkNowhere;
      what[u] = j < chunk ? m[1] : 0u;
      if constexpr (sizeof(GT) == 2) rows[u] = __builtin_amdgcn_raw_buffer_load_b64(ry, y + col_y, 0, aux);
      else rows[u] = __builtin_amdgcn_raw_buffer_load_b128(ry, y + col_y, 0, aux);
      if ((what[u] & kStore) != 0) old[u] = __builtin_amdgcn_raw_buffer_load_b128(rw, (what[u] & ~kFlags) + col_w, 0, BAGGED ? kNonTemporal : 0);
    };
    auto step = [&](int j, int u) __attribute__((always_inline)) {
      float v[4];
      if constexpr (sizeof(GT) == 2) {
        v[0] = __uint_as_float(rows[u][0] << 16);
        v[1] = __uint_as_float(rows[u][0] & 0xffff0000u);
        v[2] = __uint_as_float(rows[u][1] << 16);
        v[3] = __uint_as_float(rows[u][1] & 0xffff0000u);
      } else {
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = __uint_as_float(rows[u][e]);
      }
      uint32_t const w = what[u];
#pragma unroll
      for (int e = 0; e < 4; e++) acc[e] += v[e];
      if ((w & kStore) != 0) {
        u32x4 sum;
#pragma unroll
        for (int e = 0; e < 4; e++) sum[e] = __float_as_uint(__uint_as_float(old[u][e]) + acc[e] * a.scale);
        __builtin_amdgcn_raw_buffer_store_b128(sum, rw, (w & ~kFlags) + col_w, 0, BAGGED ? kNonTemporal : 0);
      }
      if ((w & kPartial) != 0) {
        *reinterpret_cast<f32x4 *>(emb_part + (2 * q + ((w & kHead) != 0 ? 0 : 1)) * PW + l * 4) = f32x4{acc[0], acc[1], acc[2], acc[3]};
      }
#pragma unroll
      for (int e = 0; e < 4; e++) acc[e] = (w & kEnds) != 0 ? 0.0f : acc[e];
      // this slot is free now: position j + DEPTH goes into it
      prefetch(j + DEPTH, u);
    };
#pragma unroll
    for (int u = 0; u < DEPTH; u++) prefetch(u, u);
#pragma unroll 1
    for (int j = 0; j < chunk; j += DEPTH) {
#pragma unroll
      for (int u = 0; u < DEPTH; u++) step(j + u, u);
    }
  }
  __syncthreads();
  if (col >= (uint32_t)a.dim) return;
  // Merge the border partials.  A run that crosses walkers has one partial per walker: the one
  // it starts in (slot 2w+1, or slot 0 if it comes from the workgroup before) and slot 2w of
  // each walker it reaches.  The walker of the first adds them up in position order, all runs
  // side by side.
  for (int s = q == 0 ? 0 : 2 * q + 1; s <= 2 * q + 1; s++) {
    int flags = part_valid[s];
    if (flags == 0) continue;
    uint32_t const id = part_id[s];
    f32x4 acc = *reinterpret_cast<f32x4 const *>(emb_part + s * PW + l * 4);
    for (int nxt = (s | 1) + 1; nxt < 2 * WALKERS && part_valid[nxt] != 0 && part_id[nxt] == id; nxt += 2) {
      flags |= part_valid[nxt];
      acc += *reinterpret_cast<f32x4 const *>(emb_part + nxt * PW + l * 4);
    }
    float *const dst = dW + (int64_t)id * a.dim + col;
    if ((flags & 6) != 0) {
#pragma unroll
      for (int e = 0; e < 4; e++) atomicAdd(dst + e, acc[e] * a.scale);
    } else {
      f32x4 const before = *reinterpret_cast<f32x4 const *>(dst);
      *reinterpret_cast<f32x4 *>(dst) = f32x4{before[0] + acc[0] * a.scale, before[1] + acc[1] * a.scale,
                                              before[2] + acc[2] * a.scale, before[3] + acc[3] * a.scale};
    }
  }
}

template <typename GT, int LPR>
static hipError_t embedding_walk_launch(hipStream_t st, WalkArgs a, GT const *dy, float *dw) {
  using Shape = WalkShape<GT, LPR>;
  int64_t const groups = ceil_div(a.dim, LPR * 4), per_wave = 64 / LPR;
  // The shortest chunk that makes no more than so many waves, half as many at the shortest (always 16 positions
  // and more: 3-5% slower below 16 384 lookups; 8 up to all of kWalkWaves: 52 us for 55 139 x 328 bf16, 46 so)
  a.chunk_shift = 3;
  while ((1 << a.chunk_shift) < Shape::kMaxChunk &&
         (a.n * groups >> a.chunk_shift) > (a.chunk_shift == 3 ? kWalkWaves / 2 : kWalkWaves) * per_wave) {
    a.chunk_shift++;
  }
  dim3 const grid((unsigned)ceil_div(a.n, (int64_t)Shape::kWalkers << a.chunk_shift), (unsigned)groups);
  auto kern = a.bag > 1 ? embedding_bwd_walk_kernel<GT, LPR, true> : embedding_bwd_walk_kernel<GT, LPR, false>;
  kern<<<grid, Shape::kThreads, 0, st>>>(a, dy, dw);
  return hipGetLastError();
}

// dim % 4 == 0, both tensors 16-byte aligned and below kWalkNowhere bytes, columns of one grid row each.
template <typename GT>
static hipError_t embedding_walk(hipStream_t st, WalkArgs const &a, GT const *dy, float *dw) {
  if (a.dim > 128) return embedding_walk_launch<GT, 64>(st, a, dy, dw);
  if (a.dim > 64) return embedding_walk_launch<GT, 32>(st, a, dy, dw);
  if (a.dim > 32) return embedding_walk_launch<GT, 16>(st, a, dy, dw);
  if (a.dim > 16) return embedding_walk_launch<GT, 8>(st, a, dy, dw);
  return embedding_walk_launch<GT, 4>(st, a, dy, dw);
}

}  // namespace ffk
