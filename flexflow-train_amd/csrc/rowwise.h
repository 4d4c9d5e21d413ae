// Row-wise reduction scaffolding shared by LayerNorm and Softmax.
//
// A row of N elements is owned by LANES lanes: by 16 or 32 where that many 16-byte vectors hold it (four or
// two rows a wavefront: the instructions of a row, which are what such kernels are bound by, are issued for
// all of them at once; [236881, 254] bf16, LayerNorm forward and backward, with a wavefront a row 249 and 469
// us, so and with the last vector below 58 and 69; Softmax 130 and 188, 38 and 60), by one wavefront (no LDS, no barrier), or by the four wavefronts of a workgroup (256).  Each lane
// keeps EPT vectors of the row in registers, so every element is read from HBM exactly once.
#pragma once
#include "ffk_common.h"

namespace ffk {

constexpr int kRowThreads = 256;

template <int LANES>
struct RowReducer {
  // smem: 2 phases x 4 waves x 2 values
  float (*smem)[4][2];
  int phase;
  __device__ __forceinline__ RowReducer(float (*s)[4][2]) : smem(s), phase(0) {}

  __device__ __forceinline__ static float lanes_sum(float v) {
    return wave_reduce<LANES < 64 ? LANES : 64>(v, [](float a, float b) { return a + b; });
  }
  __device__ __forceinline__ void sum2(float &a, float &b) {
    a = lanes_sum(a);
    b = lanes_sum(b);
    if (LANES > 64) {
      int const wave = threadIdx.x >> 6;
      if ((threadIdx.x & 63) == 0) {
        smem[phase][wave][0] = a;
        smem[phase][wave][1] = b;
      }
      __syncthreads();
      a = smem[phase][0][0] + smem[phase][1][0] + smem[phase][2][0] + smem[phase][3][0];
      b = smem[phase][0][1] + smem[phase][1][1] + smem[phase][2][1] + smem[phase][3][1];
      phase ^= 1;
    }
  }
  __device__ __forceinline__ float sum(float a) {
    float b = 0.0f;
    sum2(a, b);
    return a;
  }
  __device__ __forceinline__ float max(float a) {
    a = wave_reduce<LANES < 64 ? LANES : 64>(a, [](float x, float y) { return fmaxf(x, y); });
    if (LANES > 64) {
      int const wave = threadIdx.x >> 6;
      if ((threadIdx.x & 63) == 0) {
        smem[phase][wave][0] = a;
      }
      __syncthreads();
      a = fmaxf(fmaxf(smem[phase][0][0], smem[phase][1][0]),
                fmaxf(smem[phase][2][0], smem[phase][3][0]));
      phase ^= 1;
    }
    return a;
  }
};

// Vector v of a row of N elements in a kernel that gives every lane one, also lanes past the row's end.
// Rows of whole aligned vectors (ANY false) are read by the lanes that have a vector, the others hold zeros.
// Otherwise a vector that would reach past the end is the row's last 16 bytes instead, so that a load is one
// instruction without a branch (element by element it is a chain of guarded loads, which every wave waits for:
// [17225, 127] bf16, LayerNorm backward 26 us and 8): its first spare() elements belong to the vector before, hold the same values
// there, and are left out of sums.  They may be stored by both, which write the same bits, but not where the
// store adds to what is there.
// STREAM: past the caches (whole vectors only).  It is a template argument because of two accesses to one
// address that differ in nothing but the hint the compiler makes one, without the hint, also where the choice
// between them is a constant.
template <typename T, bool ANY, int EPT, int LANES>
struct LaneRow {
  static constexpr int V = VecIO<T>::kVec;
  // only the narrowest form is chosen for rows shorter than a vector
  static constexpr bool kMayBeShort = ANY && EPT == 1 && LANES == 16;
  __host__ __device__ static __forceinline__ int count(int N) { return ANY ? (N + V - 1) / V : N / V; }
  __device__ static __forceinline__ int spare(int v, int N) { return min(max((v + 1) * V - N, 0), V); }
  // whether some lane's vector j may have spare elements (the same in every lane)
  __device__ static __forceinline__ bool ragged(int j, int N) { return ANY && (EPT == 1 || (j + 1) * LANES * V > N); }
  // (v >= 0; ANY needs N >= V unless kMayBeShort)
  template <bool STREAM = false>
  __device__ static __forceinline__ u32x4 load_raw(T const *row, int v, int N) {
    if constexpr (ANY) {
      if (kMayBeShort && N < V) {
        float x[V];
#pragma unroll
        for (int e = 0; e < V; e++) x[e] = e >= V - N ? VecIO<T>::load1(row + e - (V - N)) : 0.0f;
        return pack_raw(x, (T const *)nullptr);
      }
      return load_raw_any(row + min(v * V, N - V));
    } else {
      u32x4 r = {0u, 0u, 0u, 0u};
      if (v < N / V) {
        if constexpr (STREAM) {
          r = load_raw_stream(row + (int64_t)v * V);
        } else {
          r = *reinterpret_cast<u32x4 const *>(row + (int64_t)v * V);
        }
      }
      return r;
    }
  }
  template <bool STREAM = false>
  __device__ static __forceinline__ void load(T const *row, int v, int N, float (&x)[V]) {
    unpack_raw(load_raw<STREAM>(row, v, N), x, (T const *)nullptr);
  }
  // OWN: not the spare elements
  template <bool STREAM = false, bool OWN = false>
  __device__ static __forceinline__ void store(T *row, int v, int N, float const (&x)[V]) {
    if (v >= count(N)) return;
    if constexpr (ANY) {
      if (OWN || (kMayBeShort && N < V)) {
        int const s = spare(v, N);
#pragma unroll
        for (int e = 0; e < V; e++) {
          if (e >= s) VecIO<T>::store1(row + v * V + e - s, x[e]);
        }
      } else {
        store_raw_any(row + min(v * V, N - V), pack_raw(x, (T const *)nullptr));
      }
    } else if constexpr (STREAM) {
      __builtin_nontemporal_store(pack_raw(x, (T const *)nullptr), reinterpret_cast<u32x4 *>(row + (int64_t)v * V));
    } else {
      *reinterpret_cast<u32x4 *>(row + (int64_t)v * V) = pack_raw(x, (T const *)nullptr);
    }
  }
};

// Which of a workgroup's rows a thread has a part in, and which lane of the row it is.  Constants, or the thread's index,
// where a row takes the whole workgroup: its addresses are then uniform (as quotients they were held per lane, and
// LayerNorm's backward, 8 vectors a lane, took 226 accumulation registers more instead of 57: [3000, 4544] fp32 48 us, 34
// so, [3000, 8192] bf16 50 and 35).
template <int LANES, int THREADS>
__device__ __forceinline__ int row_in_block() {
  return LANES == THREADS ? 0 : threadIdx.x / LANES;
}
template <int LANES, int THREADS>
__device__ __forceinline__ int lane_in_row() {
  return LANES == THREADS ? threadIdx.x : threadIdx.x % LANES;
}

// Picks (EPT, LANES) for a row of `nvec` 16-byte vectors; returns false when the
// row does not fit in registers (nvec > 256 * 8).
// whole: rows of whole aligned vectors.  A workgroup, two vectors a lane, takes rows that a wave would need eight a
// lane for, where it has few idle lanes.  Softmax forward / backward, us, and in brackets by waves: bf16 [16384, 4096] 47 / 62
// (51 / 67), [16384, 3600] 43 / 59 (51 / 59), [3001, 3600] 8.9 / 10.6 (9.6 / 10.5), fp32 [16384, 1800] 43 / 59 (54 / 60), [8192,
// 1537] 18.5 / 28.5 (19.3 / 29.5).  Not fp32 rows that fill the wave ([8192, 2048] 24.9 / 36.7 (23.2 / 39.8)), nor bf16 rows at any
// address ([16384, 3073] 41 / 62 (38 / 55)), nor rows of few more vectors than 256 (bf16 [16384, 2060] 29.3 / 36.9 (27.1 / 38.3)).
static inline bool pick_row_config(int64_t nvec, size_t elem_size, bool whole, int &ept, int &lanes) {
  if (nvec > 320 && (elem_size == 2 ? whole && nvec <= 512 : nvec <= 480)) {
    lanes = 256;
    ept = 2;
    return true;
  }
  if (nvec <= 64 * 8) {
    lanes = nvec <= 16 ? 16 : nvec <= 32 ? 32 : 64;
    ept = nvec <= 64 ? 1 : nvec <= 128 ? 2 : nvec <= 256 ? 4 : 8;
    return true;
  }
  if (nvec <= 256 * 8) {
    lanes = 256;
    ept = nvec <= 256 * 4 ? 4 : 8;
    return true;
  }
  return false;
}

// The LayerNorm kernels': at most one wave per row up to 128 vectors, or up to 64 * wave_vectors of them,
// one workgroup per row beyond (few vectors per lane keeps register use low and
// measured 76% vs 59% of HBM peak for a [16384, 4096] bf16 LayerNorm forward).
static inline bool pick_row_config_small(int64_t nvec, int wave_vectors, int &ept, int &lanes) {
  if (nvec <= 64 * wave_vectors) {
    lanes = nvec <= 16 ? 16 : nvec <= 32 ? 32 : 64;
    ept = nvec <= 64 ? 1 : (int)((nvec + 63) / 64);
    return true;
  }
  if (nvec <= 256 * 8) {
    lanes = 256;
    ept = nvec <= 256 ? 1 : nvec <= 512 ? 2 : nvec <= 1024 ? 4 : 8;
    return true;
  }
  return false;
}

// Rows of 129 to 256 vectors leave up to half of a workgroup's lanes idle, and pass a barrier for each sum, where a
// wave takes them in three or four vectors a lane.  The wave's form and, in brackets, the workgroup's:
//   forward, 129-192 vectors: [60000, 513] fp32 46 us (67), [32768, 768] 41 (42), [3001, 640] 5.1 (5.8); bf16
//     [60000, 1025] 61 (106), [32768, 1536] 43 (56), [4096, 1280] 6.4 (7.8)
//   forward, 193-256 vectors: bf16 [32768, 1800] 54 (61), [16384, 2048] 30 (34), [3001, 2048] 7.7 (7.6); but fp32
//     [32768, 1000] 54 (48), whose workgroup has fewer idle lanes than its rows have bytes
template <typename T>
constexpr int ln_fwd_wave_vectors() { return sizeof(T) == 2 ? 4 : 3; }
//   backward, 129-192 vectors: [60000, 513] fp32 74 (126), [16384, 768] 35 (42), [6000, 768] 15.0 (15.2); bf16 [60000, 1025]
//     76 (148), [16384, 1280] 32 (44), [6000, 1536] 17.1 (17.4); but [4096, 768] 12.9 (12.4), bf16 [4096, 1280] 14.7
//     (13.5): waves of few rows each, whose sums of the parameters' gradients have yet to be folded
//   backward, 193-256 vectors: bf16 [16384, 2048] 52 (47), fp32 [4096, 1024] 15 (14): registers
inline int ln_bwd_wave_vectors(int64_t rows) { return rows >= 6000 ? 3 : 2; }

#define FFK_ROW_DISPATCH_SMALL(EPT_, LANES_, CALL)                             \
  do {                                                                         \
    if ((LANES_) == 16) {                                                      \
      CALL(1, 16);                                                             \
    } else if ((LANES_) == 32) {                                               \
      CALL(1, 32);                                                             \
    } else if ((LANES_) == 64) {                                               \
      if ((EPT_) == 1) { CALL(1, 64); }                                        \
      else if ((EPT_) == 2) { CALL(2, 64); }                                   \
      else { CALL(3, 64); }                                                    \
    } else {                                                                   \
      if ((EPT_) == 1) { CALL(1, 256); }                                       \
      else if ((EPT_) == 2) { CALL(2, 256); }                                  \
      else if ((EPT_) == 4) { CALL(4, 256); }                                  \
      else { CALL(8, 256); }                                                   \
    }                                                                          \
  } while (0)

// (and of T where a wave takes four vectors a lane)
#define FFK_ROW_DISPATCH_FORWARD(EPT_, LANES_, CALL)                           \
  do {                                                                         \
    if ((LANES_) == 64 && (EPT_) == 4) {                                       \
      if constexpr (ln_fwd_wave_vectors<T>() == 4) { CALL(4, 64); }            \
    } else {                                                                   \
      FFK_ROW_DISPATCH_SMALL(EPT_, LANES_, CALL);                              \
    }                                                                          \
  } while (0)

#define FFK_ROW_DISPATCH(EPT_, LANES_, CALL)                                   \
  do {                                                                         \
    if ((LANES_) == 16) {                                                      \
      CALL(1, 16);                                                             \
    } else if ((LANES_) == 32) {                                               \
      CALL(1, 32);                                                             \
    } else if ((LANES_) == 64) {                                               \
      if ((EPT_) == 1) { CALL(1, 64); }                                        \
      else if ((EPT_) == 2) { CALL(2, 64); }                                   \
      else if ((EPT_) == 4) { CALL(4, 64); }                                   \
      else { CALL(8, 64); }                                                    \
    } else {                                                                   \
      if ((EPT_) == 2) { CALL(2, 256); }                                       \
      else if ((EPT_) == 4) { CALL(4, 256); }                                  \
      else { CALL(8, 256); }                                                   \
    }                                                                          \
  } while (0)

}  // namespace ffk
