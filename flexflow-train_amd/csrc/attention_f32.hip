// Fused (flash-style) attention for gfx950 in fp32: the core behind the
// reference's own MultiHeadAttention signature, which hands float tensors to
// cudnnMultiHeadAttnForward / BackwardData (lib/kernels/src/cuda/ops/
// attention_kernels.cu:224,261).  Same scheme as the bf16 core in
// attention.hip -- scores never leave the CU, a lane owns one query row of the
// transposed score tile, the backward is two kernels without atomics -- on the
// fp32 matrix instruction v_mfma_f32_32x32x2f32:
//   A operand: lane l holds A[row l%32][k = l/32]
//   B operand: lane l holds B[k = l/32][column l%32]
//   accumulator element r of lane l: row 8*(r/4) + 4*(l/32) + r%4, column l%32.
// A contraction over the head dim takes DP/2 steps; the lanes of half h = l/32
// walk d = h*DP/2 + step, so both halves read contiguous floats (16-byte LDS
// reads, four steps each).  A contraction over keys or queries re-uses an
// accumulator tile as an operand: step r takes element r of every lane, whose
// reduction index is 8*(r/4) + 4*h + r%4, and the other operand is read from
// the LDS tile row of that index.
// head sizes: any multiple of 4 up to 256, and the value head size (V, O, dO,
// dV) may differ from the query/key one (Q, K, dQ, dK): the reference's model
// builders ask for kdim = vdim = 256 (lib/models/src/models/transformer/
// transformer.cc:37-38, bert/bert.cc:64-65) and the projection sizes are free
// (lib/op-attrs/src/op-attrs/ops/attention.cc:23-37).  DP is the larger of
// the two rounded up to 32, 64, 128 or 256; the missing columns of either
// kind are read as zeros.  At DP = 256 a wave's operands and accumulators no
// longer fit its 512 registers in one pass of the backward: there two waves
// share their rows (the pair kernels), and tiles go straight to LDS.
#include "ffk_common.h"
#include "lds_dma.h"
#include "fused_ops.h"
#include <algorithm>
#include <type_traits>

namespace ffk {

constexpr float kLog2eF = 1.4426950408889634f;
constexpr float kLn2F = 0.6931471805599453f;

struct AttnF32Params {
  float const *q, *k, *v, *o, *d_o;
  float *out;  // forward: O
  float *lse;  // forward: written; backward: read
  float *delta;
  float *dq, *dk, *dv;
  int B, H, Sq, Skv, Dq, Dv;  // Dq: head size of Q, K, dQ, dK; Dv: of V, O, dO, dV
  int64_t q_bs, q_ss, k_bs, k_ss, v_bs, v_ss, o_bs, o_ss;
  float scale, scale_log2;
  int causal;
  // The pairs of batch entry and head that a launch of the backward takes, and where dK and dV's kernel leaves dS
  // for dQ's (nullptr: it does not): [pairs][Sq][ds_ld], rows of whole tiles of 32 keys.
  int pair0, pairs;
  float *ds;
  int ds_ld;
};

template <int DP>
struct AttnF32Cfg {
  static constexpr int kBlk = 128;        // rows a workgroup owns
  static constexpr int kTile = 32;        // rows of the streamed operands per step
  static constexpr int kStrideA = DP + 4; // tile read along d only (16-byte reads, conflict-free)
  static constexpr int kStrideB = DP + 8; // tile also read one row per half-wave: 4 rows apart = 32 banks apart
  static constexpr int kChunks = kTile * DP / 4 / 256;  // 16-byte chunks per thread
  static_assert(kTile * DP / 4 % 256 == 0, "tile chunks");
  // next tile fetched into registers while this one is computed on (not at DP = 256: no room)
  static constexpr bool kPrefetch = DP <= 128;
};

// DP = 256: the next tile goes straight to LDS while this one is computed on, a row (64 lanes of 16
// bytes) per instruction.  With one wave per SIMD nothing else covers the loads: without it every
// 32-row tile waited for its rows (batch 8 x 8 heads x 512: forward 176 -> 172 us).
// `rsrc`: the operand's rows of this (batch, head); lanes beyond its head size D read zeros (their
// offset lies past any bound).  Row offsets fit 31 bits (checked on the host).
constexpr unsigned kRowsBound = 0x80000000u;
__device__ __forceinline__ unsigned row_lane_offset(int lane, int D) {
  return lane * 4 < D ? (unsigned)lane * 16u : kRowsBound;
}
template <int STRIDE>
__device__ __forceinline__ void tile_dma(i32x4 rsrc, unsigned lane_off, int64_t row_stride, int row0, int last_row,
                                         int wave, float *tile) {
  unsigned const lds = lds_address_of(tile);
#pragma unroll
  for (int i = 0; i < 8; i++) {
    int const row = wave * 8 + i;
    lds_dma16(rsrc, lane_off, (unsigned)min(row0 + row, last_row) * (unsigned)(row_stride * 4),
              lds + (unsigned)(row * STRIDE * 4));
  }
}

__device__ __forceinline__ f32x4 load4_or_zero(float const *row, int d0, int D) {
  f32x4 z = {0.0f, 0.0f, 0.0f, 0.0f};
  return d0 < D ? *reinterpret_cast<f32x4 const *>(row + d0) : z;
}

// This lane's row of an owned operand, in the step order of the d contraction.
template <int DP>
__device__ __forceinline__ void load_owned_row(float const *row, int D, int h32, float (&f)[DP / 2]) {
#pragma unroll
  for (int c = 0; c < DP / 8; c++) {
    f32x4 x = load4_or_zero(row, h32 * (DP / 2) + 4 * c, D);
    f[4 * c] = x[0];
    f[4 * c + 1] = x[1];
    f[4 * c + 2] = x[2];
    f[4 * c + 3] = x[3];
  }
}

// Streamed tile: global -> registers, registers -> LDS.
template <int DP, int N>
__device__ __forceinline__ void tile_gload(float const *base, int64_t row_stride, int row0, int last_row, int D,
                                           int t, f32x4 (&r)[N]) {
#pragma unroll
  for (int i = 0; i < N; i++) {
    int const c = t + i * 256;
    int const row = c / (DP / 4), ch = c % (DP / 4);
    int const gr = min(row0 + row, last_row);
    r[i] = load4_or_zero(base + (int64_t)gr * row_stride, ch * 4, D);
  }
}
template <int DP, int STRIDE, int N>
__device__ __forceinline__ void tile_lstore(float *tile, int t, f32x4 const (&r)[N]) {
#pragma unroll
  for (int i = 0; i < N; i++) {
    int const c = t + i * 256;
    int const row = c / (DP / 4), ch = c % (DP / 4);
    *reinterpret_cast<f32x4 *>(tile + row * STRIDE + ch * 4) = r[i];
  }
}

// acc (+)= T . owned^T over d: rows = the tile's rows, columns = the owned rows
// of this wave (one per lane and half).  tile_lane = tile + (l%32)*stride + h*DP/2.
// Both contractions read the LDS fragments of a group of matrix instructions under the group before
// it (at least four of 64 cycles each), held there by scheduling barriers: with one or two waves to
// a SIMD nothing else covers the LDS latency, and the compiler left alone puts every read right in
// front of the two instructions that use it.  Head size 256, batch 8 x 8 heads x 512: forward 172 -> 167
// us, dK/dV 359 -> 345, dQ 278 -> 273.
template <int DP>
__device__ __forceinline__ void contract_d(float const *tile_lane, float const (&owned)[DP / 2], f32x16 &acc) {
  constexpr int N = DP / 8, G = 2;
  f32x4 a[2][G];
#pragma unroll
  for (int g = 0; g < G; g++) a[0][g] = *reinterpret_cast<f32x4 const *>(tile_lane + 4 * g);
#pragma unroll
  for (int c = 0; c < N; c += G) {
    if (c + G < N) {
#pragma unroll
      for (int g = 0; g < G; g++) {
        a[(c / G + 1) & 1][g] = *reinterpret_cast<f32x4 const *>(tile_lane + 4 * (c + G + g));
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < G; g++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[(c / G) & 1][g][e], owned[4 * (c + g) + e], acc, 0, 0, 0);
      }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// acc[i] += (columns 32 i .. of the tile's rows) x (score tile), over the tile's 32 rows.  The score
// tile is an accumulator's 16 elements per lane; step r takes the rows 8*(r/4) + 4*h + r%4.
// tile_lane = tile + 4*h*STRIDE + l%32.  TILE_A: the tile is the A operand (rows of the result =
// its columns), otherwise the B operand.
template <int N, int STRIDE, bool TILE_A>
__device__ __forceinline__ void contract_rows(float const *tile_lane, float const (&score)[16], f32x16 (&acc)[N]) {
  constexpr int G = N >= 8 ? 1 : N >= 4 ? 2 : 4;
  float f[2][G][N];
  auto read = [&](int r0, float (&d)[G][N]) {
#pragma unroll
    for (int g = 0; g < G; g++) {
      int const row = 8 * ((r0 + g) >> 2) + ((r0 + g) & 3);
#pragma unroll
      for (int i = 0; i < N; i++) d[g][i] = tile_lane[row * STRIDE + i * 32];
    }
  };
  read(0, f[0]);
#pragma unroll
  for (int r = 0; r < 16; r += G) {
    if (r + G < 16) read(r + G, f[(r / G + 1) & 1]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < G; g++)
#pragma unroll
      for (int i = 0; i < N; i++) {
        float const t = f[(r / G) & 1][g][i];
        acc[i] = TILE_A ? __builtin_amdgcn_mfma_f32_32x32x2f32(t, score[r + g], acc[i], 0, 0, 0)
                        : __builtin_amdgcn_mfma_f32_32x32x2f32(score[r + g], t, acc[i], 0, 0, 0);
      }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// A wave's accumulators to LDS and back, for the wave that adds them up: 16 bytes a lane, lanes side by side.
template <int NI>
__device__ __forceinline__ void acc_put(float *to, f32x16 const (&acc)[NI], int lane) {
#pragma unroll
  for (int i = 0; i < NI; i++)
#pragma unroll
    for (int g = 0; g < 4; g++)
      *reinterpret_cast<f32x4 *>(to + ((i * 4 + g) * 64 + lane) * 4) =
          f32x4{acc[i][4 * g], acc[i][4 * g + 1], acc[i][4 * g + 2], acc[i][4 * g + 3]};
}
template <int NI>
__device__ __forceinline__ void acc_add(float const *from, float factor, f32x16 (&acc)[NI], int lane) {
#pragma unroll
  for (int i = 0; i < NI; i++)
#pragma unroll
    for (int g = 0; g < 4; g++) {
      f32x4 const x = *reinterpret_cast<f32x4 const *>(from + ((i * 4 + g) * 64 + lane) * 4);
#pragma unroll
      for (int e = 0; e < 4; e++) acc[i][4 * g + e] += x[e] * factor;
    }
}

// --------------------------------------------------------------------------
// forward: workgroup = 128 / KW query rows of one (batch, head), 32 per group of KW waves, which take the keys of a
// step of 32 * KW in turn and add up in LDS at the end (for problems that would leave CUs without a workgroup)
// --------------------------------------------------------------------------
template <int DP, int KW>
struct AttnF32Fwd {
  using C = AttnF32Cfg<DP>;
  static constexpr int kT = 32 * KW, kK = kT * C::kStrideA, kV = kT * C::kStrideB;  // rows of a step, floats of its tiles
  static constexpr int kBuffers = 2 * (kK + kV) * 4 <= 150 * 1024 ? 2 : 1;
  static constexpr int kSlot = DP * 32 + 128, kMerge = (KW - 1) * (4 / KW) * kSlot;
  static constexpr int kFloats = kBuffers * (kK + kV) > kMerge ? kBuffers * (kK + kV) : kMerge;
  static constexpr int kChunks = kT * DP / 4 / 256;
};
template <int DP, bool DMA, int KW>
__global__ __launch_bounds__(256) void attn_f32_fwd_kernel(AttnF32Params p) {
  using C = AttnF32Cfg<DP>;
  using F = AttnF32Fwd<DP, KW>;
  static_assert(KW == 1 || (C::kPrefetch && !DMA), "the split form prefetches into registers");
  constexpr int T = F::kT, QR = 128 / KW;
  __shared__ __attribute__((aligned(16))) float pool[F::kFloats];
  auto Ks = [&](int buf) __attribute__((always_inline)) { return pool + (F::kBuffers == 2 ? buf : 0) * F::kK; };
  auto Vs = [&](int buf) __attribute__((always_inline)) { return pool + F::kBuffers * F::kK + (F::kBuffers == 2 ? buf : 0) * F::kV; };
  int const t = threadIdx.x, lane = t & 63, h32 = lane >> 5, l32 = lane & 31;
  int const wave = __builtin_amdgcn_readfirstlane(t >> 6);
  int const qw = wave / KW, kw = wave % KW;
  int const nqb = (p.Sq + QR - 1) / QR;
  int const hb = blockIdx.x % (p.H * p.B);
  int const qb = nqb - 1 - blockIdx.x / (p.H * p.B);  // heaviest causal blocks first
  int const head = hb % p.H, b = hb / p.H;
  int const q0 = qb * QR, qw0 = q0 + qw * 32;
  int const qrow = qw0 + l32;
  float const *qp = p.q + (int64_t)b * p.q_bs + (int64_t)head * p.Dq;
  float const *kp = p.k + (int64_t)b * p.k_bs + (int64_t)head * p.Dq;
  float const *vp = p.v + (int64_t)b * p.v_bs + (int64_t)head * p.Dv;

  float qf[DP / 2];
  load_owned_row<DP>(qp + (int64_t)min(qrow, p.Sq - 1) * p.q_ss, p.Dq, h32, qf);

  int kv_end = p.Skv;
  if (p.causal) kv_end = min(p.Skv, q0 + QR);
  int const ntiles = (kv_end + T - 1) / T;

  f32x16 oacc[DP / 32];
#pragma unroll
  for (int i = 0; i < DP / 32; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) oacc[i][r] = 0.0f;
  float m_run = -INFINITY, l_run = 0.0f;

  f32x4 rk[F::kChunks], rv[F::kChunks];
  i32x4 k_rsrc, v_rsrc;
  unsigned k_lane = 0, v_lane = 0;
  if constexpr (DMA) {
    k_rsrc = buffer_resource(kp, kRowsBound);
    v_rsrc = buffer_resource(vp, kRowsBound);
    k_lane = row_lane_offset(lane, p.Dq);
    v_lane = row_lane_offset(lane, p.Dv);
  }
  auto fetch = [&](int kv0, int buf) {
    if constexpr (DMA) {
      tile_dma<C::kStrideA>(k_rsrc, k_lane, p.k_ss, kv0, p.Skv - 1, wave, Ks(buf));
      tile_dma<C::kStrideB>(v_rsrc, v_lane, p.v_ss, kv0, p.Skv - 1, wave, Vs(buf));
    } else {
      tile_gload<DP>(kp, p.k_ss, kv0, p.Skv - 1, p.Dq, t, rk);
      tile_gload<DP>(vp, p.v_ss, kv0, p.Skv - 1, p.Dv, t, rv);
    }
  };
  auto stash = [&](int buf) {
    if constexpr (DMA) {
      wait_vmcnt<0>();
    } else {
      tile_lstore<DP, C::kStrideA>(Ks(buf), t, rk);
      tile_lstore<DP, C::kStrideB>(Vs(buf), t, rv);
    }
  };
  fetch(0, 0);
  stash(0);
  if constexpr (DMA) wait_all_vmem_known_to_compiler();
  __syncthreads();
  int cur = 0;
  for (int it = 0; it < ntiles; it++) {
    int const kv0 = it * T + kw * 32;  // this wave's keys
    bool const more = it + 1 < ntiles;
    if ((DMA || C::kPrefetch) && more) fetch((it + 1) * T, cur ^ 1);
    // a wave whose rows all lie before its keys (causal), or whose keys do not exist, has nothing to add
    bool const active = (KW == 1 || kv0 < p.Skv) && (!p.causal || kv0 <= qw0 + 31);
    if (active) {
      // S^T: rows = keys of the tile, column = this lane's query
      f32x16 s;
#pragma unroll
      for (int r = 0; r < 16; r++) s[r] = 0.0f;
      contract_d<DP>(Ks(cur) + (kw * 32 + l32) * C::kStrideA + h32 * (DP / 2), qf, s);
      bool const need_mask = (kv0 + C::kTile > p.Skv) || (p.causal && kv0 + C::kTile - 1 > qw0);
      if (need_mask) {
#pragma unroll
        for (int r = 0; r < 16; r++) {
          int const kv = kv0 + 8 * (r >> 2) + 4 * h32 + (r & 3);
          if (kv >= p.Skv || (p.causal && kv > qrow)) s[r] = -INFINITY;
        }
      }
      float mx = -INFINITY;
#pragma unroll
      for (int r = 0; r < 16; r++) mx = fmaxf(mx, s[r]);
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64)) * p.scale_log2;
      // one wave of a group: finite from the first tile on, key 0 is visible to every query.  Of several, one may so
      // far have met masked keys alone: its maximum stays -inf, and what it subtracts is 0 instead.
      float const m_new = fmaxf(m_run, mx);
      float const m_sub = KW > 1 && m_new == -INFINITY ? 0.0f : m_new;
      float const alpha = __builtin_amdgcn_exp2f(m_run - m_sub);
      float sum = 0.0f;
      float pv[16];
#pragma unroll
      for (int r = 0; r < 16; r++) {
        pv[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], p.scale_log2, -m_sub));
        sum += pv[r];
      }
      sum += __shfl_xor(sum, 32, 64);
      l_run = l_run * alpha + sum;
      m_run = m_new;
      if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
#pragma unroll
        for (int i = 0; i < DP / 32; i++)
#pragma unroll
          for (int r = 0; r < 16; r++) oacc[i][r] *= alpha;
      }
      // O^T += V^T P^T: A = V^T (row d), B = P^T (column = query), reduction over keys
      contract_rows<DP / 32, C::kStrideB, true>(Vs(cur) + (kw * 32 + 4 * h32) * C::kStrideB + l32, pv, oacc);
    }
    if (F::kBuffers == 1) __syncthreads();
    if (more) {
      if (!DMA && !C::kPrefetch) fetch((it + 1) * T, cur ^ 1);
      stash(cur ^ 1);
    }
    __syncthreads();
    cur ^= 1;
  }
  if constexpr (KW > 1) {
    float *const slots = pool + qw * (KW - 1) * F::kSlot;
    if (kw > 0) {
      float *const mine = slots + (kw - 1) * F::kSlot;
      acc_put<DP / 32>(mine, oacc, lane);
      mine[DP * 32 + lane] = m_run;
      mine[DP * 32 + 64 + lane] = l_run;
    }
    __syncthreads();
    if (kw > 0) return;
    float m_all = m_run;  // finite: this wave's first keys include key 0
#pragma unroll
    for (int w = 0; w < KW - 1; w++) m_all = fmaxf(m_all, slots[w * F::kSlot + DP * 32 + lane]);
    float const mine = __builtin_amdgcn_exp2f(m_run - m_all);
    l_run *= mine;
#pragma unroll
    for (int i = 0; i < DP / 32; i++)
#pragma unroll
      for (int r = 0; r < 16; r++) oacc[i][r] *= mine;
#pragma unroll
    for (int w = 0; w < KW - 1; w++) {
      float const *const other = slots + w * F::kSlot;
      float const factor = __builtin_amdgcn_exp2f(other[DP * 32 + lane] - m_all);
      l_run += other[DP * 32 + 64 + lane] * factor;
      acc_add<DP / 32>(other, factor, oacc, lane);
    }
    m_run = m_all;
  }

  if (qrow < p.Sq) {
    float const inv = 1.0f / l_run;
    float *op = p.out + (int64_t)b * p.o_bs + (int64_t)qrow * p.o_ss + (int64_t)head * p.Dv;
#pragma unroll
    for (int i = 0; i < DP / 32; i++) {
#pragma unroll
      for (int g = 0; g < 4; g++) {
        int const d = i * 32 + 8 * g + 4 * h32;
        if (d < p.Dv) {
          f32x4 w = {oacc[i][4 * g] * inv, oacc[i][4 * g + 1] * inv, oacc[i][4 * g + 2] * inv,
                     oacc[i][4 * g + 3] * inv};
          *reinterpret_cast<f32x4 *>(op + d) = w;
        }
      }
    }
    if (h32 == 0 && p.lse != nullptr) {
      p.lse[((int64_t)b * p.H + head) * p.Sq + qrow] = (m_run + __log2f(l_run)) * kLn2F;
    }
  }
}

// delta[b,h,q] = sum_d O * dO; DP/4 lanes share a row
template <int DP>
__global__ __launch_bounds__(256) void attn_f32_delta_kernel(AttnF32Params p) {
  constexpr int LPR = DP / 4;
  constexpr int RPW = 64 / LPR;
  int const lane = threadIdx.x & 63;
  int64_t const row = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * RPW + lane / LPR;
  int64_t const total = (int64_t)p.B * p.H * p.Sq;
  float s = 0.0f;
  bool const ok = row < total;
  int head = 0, q = 0, b = 0;
  if (ok) {
    head = (int)(row % p.H);
    q = (int)((row / p.H) % p.Sq);
    b = (int)(row / ((int64_t)p.Sq * p.H));
    int64_t const off = (int64_t)b * p.o_bs + (int64_t)q * p.o_ss + (int64_t)head * p.Dv;
    int const d0 = (lane % LPR) * 4;
    f32x4 const o = load4_or_zero(p.o + off, d0, p.Dv);
    f32x4 const g = load4_or_zero(p.d_o + off, d0, p.Dv);
    s = o[0] * g[0] + o[1] * g[1] + o[2] * g[2] + o[3] * g[3];
  }
#pragma unroll
  for (int m = 1; m < LPR; m <<= 1) s += __shfl_xor(s, m, 64);
  if (ok && lane % LPR == 0) p.delta[((int64_t)b * p.H + head) * p.Sq + q] = s;
}

// A 32 x 32 tile of dS to p.ds: rows = queries from qt0 on, column = this lane's key (32 lanes write 128 bytes of a row).
// The descriptor of a pair's dS drops rows that do not exist (of up to 96 past the last, f32_pairs_at_a_time), and
// a row is a scalar multiple away from one offset, formed anew for each tile: no register more than without dS.  (With an
// address and a guard for each row, 48 registers, the kernels spilled at head size 128 and in the form for 132 to 252, and two
// waves ran on a SIMD at 32 instead of three; whole backward 1.5 to 5% longer by head size, more for the guards than for the
// spills, and with 6 x 32 heads x 333 of 20 1% longer than where dS is computed twice.)
__device__ __forceinline__ void save_scores(AttnF32Params const &p, int pair, int qt0, int key, int h32, float const (&e)[16]) {
  unsigned const step = (unsigned)p.ds_ld * 4u;  // bytes; a pair has 512 MB of them at most
  __amdgpu_buffer_rsrc_t const rsrc = __builtin_amdgcn_make_buffer_rsrc(p.ds + (int64_t)pair * p.Sq * p.ds_ld, 0, p.Sq * (int)step, 0x00020000);
  unsigned off = (unsigned)(qt0 + 4 * h32) * step + 4u * key;
  asm("" : "+v"(off));  // keeps the sixteen offsets of a tile from being kept instead of this one
#pragma unroll
  for (int r = 0; r < 16; r++) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, e[r]), rsrc, off + (8 * (r >> 2) + (r & 3)) * step, 0, 0);
  }
}

// --------------------------------------------------------------------------
// backward (A): dK, dV.  Workgroup owns 128 key rows, streams query tiles.
// Where the pair kernels are not taken (launch_f32_backward).
// --------------------------------------------------------------------------
template <int DP, bool SAVE>
__global__ __launch_bounds__(256) void attn_f32_bwd_dkdv_kernel(AttnF32Params p) {
  using C = AttnF32Cfg<DP>;
  __shared__ __attribute__((aligned(16))) float Qs[2][C::kTile * C::kStrideB];
  __shared__ __attribute__((aligned(16))) float Gs[2][C::kTile * C::kStrideB];  // dO
  __shared__ __attribute__((aligned(16))) float Ls[2][C::kTile], Ds[2][C::kTile];
  int const t = threadIdx.x, lane = t & 63, h32 = lane >> 5, l32 = lane & 31;
  int const wave = __builtin_amdgcn_readfirstlane(t >> 6);
  int const pair = blockIdx.x % p.pairs, hb = p.pair0 + pair;
  int const head = hb % p.H, b = hb / p.H;
  int const kv0 = (blockIdx.x / p.pairs) * C::kBlk;
  int const kvrow = kv0 + wave * 32 + l32;
  float const *qp = p.q + (int64_t)b * p.q_bs + (int64_t)head * p.Dq;
  float const *gp = p.d_o + (int64_t)b * p.o_bs + (int64_t)head * p.Dv;
  float const *kp = p.k + (int64_t)b * p.k_bs + (int64_t)head * p.Dq;
  float const *vp = p.v + (int64_t)b * p.v_bs + (int64_t)head * p.Dv;
  float const *lsep = p.lse + ((int64_t)b * p.H + head) * p.Sq;
  float const *delp = p.delta + ((int64_t)b * p.H + head) * p.Sq;

  float kf[DP / 2], vf[DP / 2];
  load_owned_row<DP>(kp + (int64_t)min(kvrow, p.Skv - 1) * p.k_ss, p.Dq, h32, kf);
  load_owned_row<DP>(vp + (int64_t)min(kvrow, p.Skv - 1) * p.v_ss, p.Dv, h32, vf);
  f32x16 dk[DP / 32], dv[DP / 32];
#pragma unroll
  for (int i = 0; i < DP / 32; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) {
      dk[i][r] = 0.0f;
      dv[i][r] = 0.0f;
    }

  int const q_begin = p.causal ? (kv0 / C::kTile) * C::kTile : 0;
  int const ntiles = q_begin < p.Sq ? (p.Sq - q_begin + C::kTile - 1) / C::kTile : 0;

  f32x4 rq[C::kChunks], rg[C::kChunks];
  float rl = 0.0f, rd = 0.0f;
  auto gload = [&](int qt0) {
    tile_gload<DP>(qp, p.q_ss, qt0, p.Sq - 1, p.Dq, t, rq);
    tile_gload<DP>(gp, p.o_ss, qt0, p.Sq - 1, p.Dv, t, rg);
    int const gr = min(qt0 + (t & (C::kTile - 1)), p.Sq - 1);
    rl = lsep[gr] * kLog2eF;
    rd = delp[gr];
  };
  auto lstore = [&](int buf) {
    tile_lstore<DP, C::kStrideB>(Qs[buf], t, rq);
    tile_lstore<DP, C::kStrideB>(Gs[buf], t, rg);
    if (t < C::kTile) {
      Ls[buf][t] = rl;
      Ds[buf][t] = rd * p.scale;
    }
  };
  if (ntiles > 0) {
    gload(q_begin);
    lstore(0);
  }
  __syncthreads();
  int cur = 0;
  for (int it = 0; it < ntiles; it++) {
    int const qt0 = q_begin + it * C::kTile;
    bool const more = it + 1 < ntiles;
    if (more) gload(qt0 + C::kTile);
    // a wave whose keys all lie after this query tile (causal) contributes nothing
    bool const active = !p.causal || kv0 + wave * 32 <= qt0 + C::kTile - 1;
    if (active) {
      // S = Q K^T, dP = dO V^T: rows = queries of the tile, column = this lane's key
      f32x16 s, dp;
#pragma unroll
      for (int r = 0; r < 16; r++) {
        s[r] = 0.0f;
        dp[r] = 0.0f;
      }
      contract_d<DP>(Qs[cur] + l32 * C::kStrideB + h32 * (DP / 2), kf, s);
      contract_d<DP>(Gs[cur] + l32 * C::kStrideB + h32 * (DP / 2), vf, dp);
      float pv[16], dsv[16];
#pragma unroll
      for (int r = 0; r < 16; r++) {
        int const ql = 8 * (r >> 2) + 4 * h32 + (r & 3);
        int const qg = qt0 + ql;
        float const e = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], p.scale_log2, -Ls[cur][ql]));
        bool const masked = qg >= p.Sq || kvrow >= p.Skv || (p.causal && kvrow > qg);
        pv[r] = masked ? 0.0f : e;
        // dS = P (dP - delta) scale; Ds holds delta * scale
        dsv[r] = masked ? 0.0f : e * __builtin_fmaf(dp[r], p.scale, -Ds[cur][ql]);
      }
      if (SAVE && kv0 + wave * 32 < p.Skv) save_scores(p, pair, qt0, kvrow, h32, dsv);
      // dV += P^T dO, dK += dS^T Q: A = the accumulator (row = key), B = dO / Q rows of the
      // matching query, reduction over the tile's queries
      contract_rows<DP / 32, C::kStrideB, false>(Gs[cur] + (4 * h32) * C::kStrideB + l32, pv, dv);
      contract_rows<DP / 32, C::kStrideB, false>(Qs[cur] + (4 * h32) * C::kStrideB + l32, dsv, dk);
    }
    if (more) {
      lstore(cur ^ 1);
    }
    __syncthreads();
    cur ^= 1;
  }

  // accumulator element r: key row 8*(r/4) + 4*h + r%4 of this wave's 32, column d = i*32 + l%32:
  // the 32 lanes of a half write 128 contiguous bytes of one row
  float *dkp = p.dk + (int64_t)b * p.k_bs + (int64_t)head * p.Dq;
  float *dvp = p.dv + (int64_t)b * p.v_bs + (int64_t)head * p.Dv;
#pragma unroll
  for (int i = 0; i < DP / 32; i++) {
    int const d = i * 32 + l32;
#pragma unroll
    for (int r = 0; r < 16; r++) {
      int const grow = kv0 + wave * 32 + 8 * (r >> 2) + 4 * h32 + (r & 3);
      if (grow < p.Skv) {
        if (d < p.Dq) dkp[(int64_t)grow * p.k_ss + d] = dk[i][r];
        if (d < p.Dv) dvp[(int64_t)grow * p.v_ss + d] = dv[i][r];
      }
    }
  }
}

// --------------------------------------------------------------------------
// backward (B): dQ.  Workgroup owns 128 query rows, streams key tiles.
// Where the pair kernels are not taken (launch_f32_backward).
// --------------------------------------------------------------------------
template <int DP>
__global__ __launch_bounds__(256) void attn_f32_bwd_dq_kernel(AttnF32Params p) {
  using C = AttnF32Cfg<DP>;
  __shared__ __attribute__((aligned(16))) float Ks[2][C::kTile * C::kStrideB];
  __shared__ __attribute__((aligned(16))) float Vs[2][C::kTile * C::kStrideA];
  int const t = threadIdx.x, lane = t & 63, h32 = lane >> 5, l32 = lane & 31;
  int const wave = __builtin_amdgcn_readfirstlane(t >> 6);
  int const nqb = (p.Sq + C::kBlk - 1) / C::kBlk;
  int const hb = blockIdx.x % (p.H * p.B);
  int const qb = nqb - 1 - blockIdx.x / (p.H * p.B);
  int const head = hb % p.H, b = hb / p.H;
  int const q0 = qb * C::kBlk;
  int const qrow = q0 + wave * 32 + l32;
  float const *qp = p.q + (int64_t)b * p.q_bs + (int64_t)head * p.Dq;
  float const *gp = p.d_o + (int64_t)b * p.o_bs + (int64_t)head * p.Dv;
  float const *kp = p.k + (int64_t)b * p.k_bs + (int64_t)head * p.Dq;
  float const *vp = p.v + (int64_t)b * p.v_bs + (int64_t)head * p.Dv;

  float qf[DP / 2], gf[DP / 2];
  int const rq = min(qrow, p.Sq - 1);
  load_owned_row<DP>(qp + (int64_t)rq * p.q_ss, p.Dq, h32, qf);
  load_owned_row<DP>(gp + (int64_t)rq * p.o_ss, p.Dv, h32, gf);
  float const lse2 = p.lse[((int64_t)b * p.H + head) * p.Sq + rq] * kLog2eF;
  float const delta_s = p.delta[((int64_t)b * p.H + head) * p.Sq + rq] * p.scale;
  f32x16 dq[DP / 32];
#pragma unroll
  for (int i = 0; i < DP / 32; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) dq[i][r] = 0.0f;

  int kv_end = p.Skv;
  if (p.causal) kv_end = min(p.Skv, q0 + C::kBlk);
  int const ntiles = (kv_end + C::kTile - 1) / C::kTile;

  f32x4 rk[C::kChunks], rv[C::kChunks];
  auto fetch = [&](int kt0) {
    tile_gload<DP>(kp, p.k_ss, kt0, p.Skv - 1, p.Dq, t, rk);
    tile_gload<DP>(vp, p.v_ss, kt0, p.Skv - 1, p.Dv, t, rv);
  };
  auto stash = [&](int buf) {
    tile_lstore<DP, C::kStrideB>(Ks[buf], t, rk);
    tile_lstore<DP, C::kStrideA>(Vs[buf], t, rv);
  };
  fetch(0);
  stash(0);
  __syncthreads();
  int cur = 0;
  for (int it = 0; it < ntiles; it++) {
    int const kt0 = it * C::kTile;
    bool const more = it + 1 < ntiles;
    if (more) fetch(kt0 + C::kTile);
    bool const active = !p.causal || kt0 <= q0 + wave * 32 + 31;
    if (active) {
      // S^T = K Q^T, dP^T = V dO^T: rows = keys of the tile, column = this lane's query
      f32x16 s, dp;
#pragma unroll
      for (int r = 0; r < 16; r++) {
        s[r] = 0.0f;
        dp[r] = 0.0f;
      }
      contract_d<DP>(Ks[cur] + l32 * C::kStrideB + h32 * (DP / 2), qf, s);
      contract_d<DP>(Vs[cur] + l32 * C::kStrideA + h32 * (DP / 2), gf, dp);
      float dsv[16];
#pragma unroll
      for (int r = 0; r < 16; r++) {
        int const kv = kt0 + 8 * (r >> 2) + 4 * h32 + (r & 3);
        float const e = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], p.scale_log2, -lse2));
        bool const masked = kv >= p.Skv || (p.causal && kv > qrow);
        dsv[r] = masked ? 0.0f : e * __builtin_fmaf(dp[r], p.scale, -delta_s);
      }
      // dQ^T += K^T dS^T: A = K^T (row d), B = dS^T, reduction over the tile's keys
      contract_rows<DP / 32, C::kStrideB, true>(Ks[cur] + (4 * h32) * C::kStrideB + l32, dsv, dq);
    }
    if (more) {
      stash(cur ^ 1);
    }
    __syncthreads();
    cur ^= 1;
  }

  if (qrow < p.Sq) {
    float *dqp = p.dq + (int64_t)b * p.q_bs + (int64_t)qrow * p.q_ss + (int64_t)head * p.Dq;
#pragma unroll
    for (int i = 0; i < DP / 32; i++) {
#pragma unroll
      for (int g = 0; g < 4; g++) {
        int const d = i * 32 + 8 * g + 4 * h32;
        if (d < p.Dq) {
          f32x4 w = {dq[i][4 * g], dq[i][4 * g + 1], dq[i][4 * g + 2], dq[i][4 * g + 3]};
          *reinterpret_cast<f32x4 *>(dqp + d) = w;
        }
      }
    }
  }
}

// --------------------------------------------------------------------------
// Two waves share 32 owned rows (head sizes beyond 128, and where
// launch_f32_backward says so), so that what a wave
// holds (one owned operand, at most one whole accumulator) stays in registers
// with room to spare, and exchange score tiles through LDS.  A workgroup owns
// 64 rows; wave w works on rows 32 * (w % 2) in role w / 2.  Bound by the fp32
// matrix pipe.  With a wave on its own, dK and dV took two launches (the scores
// computed in both) and dQ spilled: batch 8 x 8 heads x 512 at
// head size 256, dK and dV 498 -> 345 us, dQ 309 -> 273.  KW = 2 (f32_split):
// both pairs own the same 32 rows and take the streamed rows in turn.
// --------------------------------------------------------------------------
struct PairTile {
  f32x4 v[4][64];  // elements 4g .. 4g+3 of each lane's accumulator
};
__device__ __forceinline__ void pair_put(PairTile &x, int lane, float const (&e)[16]) {
#pragma unroll
  for (int g = 0; g < 4; g++) x.v[g][lane] = f32x4{e[4 * g], e[4 * g + 1], e[4 * g + 2], e[4 * g + 3]};
}
__device__ __forceinline__ void pair_get(PairTile const &x, int lane, float (&e)[16]) {
#pragma unroll
  for (int g = 0; g < 4; g++) {
    f32x4 const v = x.v[g][lane];
#pragma unroll
    for (int i = 0; i < 4; i++) e[4 * g + i] = v[i];
  }
}
// the waves' LDS writes before it are visible after it; direct loads in flight stay in flight
__device__ __forceinline__ void pair_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Streams two operands' tiles of T rows into two buffers each, one tile ahead: by direct loads (DMA), or
// through registers.
template <int DP, bool DMA, int STRIDE0, int STRIDE1, int T>
struct PairStream {
  static_assert(!DMA || T == 32, "direct loads are written for 32 rows");
  float const *base[2];
  int64_t ss[2];
  int D[2];
  int last, t, lane, wave;
  i32x4 rsrc[2];
  unsigned lane_off[2];
  f32x4 r0[DMA ? 1 : T * DP / 4 / 256], r1[DMA ? 1 : T * DP / 4 / 256];
  __device__ __forceinline__ void init() {
    if constexpr (DMA) {
#pragma unroll
      for (int o = 0; o < 2; o++) {
        rsrc[o] = buffer_resource(base[o], kRowsBound);
        lane_off[o] = row_lane_offset(lane, D[o]);
      }
    }
  }
  __device__ __forceinline__ void fetch(int row0, float *t0, float *t1) {
    if constexpr (DMA) {
      tile_dma<STRIDE0>(rsrc[0], lane_off[0], ss[0], row0, last, wave, t0);
      tile_dma<STRIDE1>(rsrc[1], lane_off[1], ss[1], row0, last, wave, t1);
    } else {
      tile_gload<DP>(base[0], ss[0], row0, last, D[0], t, r0);
      tile_gload<DP>(base[1], ss[1], row0, last, D[1], t, r1);
    }
  }
  __device__ __forceinline__ void land(float *t0, float *t1) const {
    if constexpr (DMA) {
      wait_vmcnt<0>();
    } else {
      tile_lstore<DP, STRIDE0>(t0, t, r0);
      tile_lstore<DP, STRIDE1>(t1, t, r1);
    }
  }
};

// dK and dV: role 0 computes S and P, hands P over and produces dV; role 1 computes dP and from
// it and P dS, and produces dK.
template <int DP, bool DMA, int KW, bool SAVE>
__global__ __launch_bounds__(256) void attn_f32_bwd_dkdv_pair_kernel(AttnF32Params p) {
  using C = AttnF32Cfg<DP>;
  constexpr int T = 32 * KW;
  __shared__ __attribute__((aligned(16))) float Qs[2][T * C::kStrideB];
  __shared__ __attribute__((aligned(16))) float Gs[2][T * C::kStrideB];  // dO
  __shared__ PairTile Ps[2];
  __shared__ __attribute__((aligned(16))) float Ls[2][T], Ds[2][T];
  int const t = threadIdx.x, lane = t & 63, h32 = lane >> 5, l32 = lane & 31;
  int const wave = __builtin_amdgcn_readfirstlane(t >> 6);
  int const blk = wave & 1, role = wave >> 1;
  int const pair = blockIdx.x % p.pairs, hb = p.pair0 + pair;
  int const head = hb % p.H, b = hb / p.H;
  int const kvg = (blockIdx.x / p.pairs) * (64 / KW);  // the workgroup's first key
  int const kv0 = KW == 1 ? kvg + blk * 32 : kvg;           // this wave's
  int const part = KW == 1 ? 0 : blk * 32;                  // its first query of a step
  int const kvrow = kv0 + l32;
  float const *lsep = p.lse + ((int64_t)b * p.H + head) * p.Sq;
  float const *delp = p.delta + ((int64_t)b * p.H + head) * p.Sq;

  float own[DP / 2];  // role 0: the row of K, role 1: of V
  {
    int const r = min(kvrow, p.Skv - 1);
    if (role == 0) load_owned_row<DP>(p.k + (int64_t)b * p.k_bs + (int64_t)head * p.Dq + (int64_t)r * p.k_ss, p.Dq, h32, own);
    else load_owned_row<DP>(p.v + (int64_t)b * p.v_bs + (int64_t)head * p.Dv + (int64_t)r * p.v_ss, p.Dv, h32, own);
  }
  f32x16 acc[DP / 32];  // role 0: dV, role 1: dK
#pragma unroll
  for (int i = 0; i < DP / 32; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) acc[i][r] = 0.0f;

  int const q_begin = p.causal ? (kvg / T) * T : 0;
  int const ntiles = q_begin < p.Sq ? (p.Sq - q_begin + T - 1) / T : 0;
  PairStream<DP, DMA, C::kStrideB, C::kStrideB, T> st;
  st.base[0] = p.q + (int64_t)b * p.q_bs + (int64_t)head * p.Dq;
  st.base[1] = p.d_o + (int64_t)b * p.o_bs + (int64_t)head * p.Dv;
  st.ss[0] = p.q_ss; st.ss[1] = p.o_ss;
  st.D[0] = p.Dq; st.D[1] = p.Dv;
  st.last = p.Sq - 1; st.t = t; st.lane = lane; st.wave = wave;
  st.init();
  float rl = 0.0f, rd = 0.0f;
  auto load_row_terms = [&](int qt0) {
    int const gr = min(qt0 + (t & (T - 1)), p.Sq - 1);
    rl = lsep[gr];
    rd = delp[gr];
  };
  auto store_row_terms = [&](int buf) {
    if (t < T) {
      Ls[buf][t] = rl * kLog2eF;
      Ds[buf][t] = rd * p.scale;
    }
  };
  if (ntiles > 0) {
    load_row_terms(q_begin);
    st.fetch(q_begin, Qs[0], Gs[0]);
    st.land(Qs[0], Gs[0]);
    store_row_terms(0);
  }
  if constexpr (DMA) wait_all_vmem_known_to_compiler();
  __syncthreads();
  int cur = 0;
  for (int it = 0; it < ntiles; it++) {
    int const step0 = q_begin + it * T, qt0 = step0 + part;
    bool const more = it + 1 < ntiles;
    if (more) {
      load_row_terms(step0 + T);
      st.fetch(step0 + T, Qs[cur ^ 1], Gs[cur ^ 1]);
    }
    // waves whose keys all lie after their queries (causal), or whose queries do not exist, contribute nothing
    bool const active = (KW == 1 || qt0 < p.Sq) && (!p.causal || kv0 <= qt0 + 31);
    float ex[16];  // role 0: P, role 1: dS
    f32x16 s;
    if (active) {
      // S = Q K^T or dP = dO V^T: rows = queries of the tile, column = this lane's key
#pragma unroll
      for (int r = 0; r < 16; r++) s[r] = 0.0f;
      contract_d<DP>((role == 0 ? Qs[cur] : Gs[cur]) + (part + l32) * C::kStrideB + h32 * (DP / 2), own, s);
      if (role == 0) {
#pragma unroll
        for (int r = 0; r < 16; r++) {
          int const ql = 8 * (r >> 2) + 4 * h32 + (r & 3);
          int const qg = qt0 + ql;
          float const e = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], p.scale_log2, -Ls[cur][part + ql]));
          bool const masked = qg >= p.Sq || kvrow >= p.Skv || (p.causal && kvrow > qg);
          ex[r] = masked ? 0.0f : e;
        }
        pair_put(Ps[blk], lane, ex);
      }
    }
    pair_barrier();
    if (active) {
      if (role == 1) {
        pair_get(Ps[blk], lane, ex);
#pragma unroll
        for (int r = 0; r < 16; r++) {
          int const ql = 8 * (r >> 2) + 4 * h32 + (r & 3);
          int const qg = qt0 + ql;
          bool const masked = qg >= p.Sq || kvrow >= p.Skv || (p.causal && kvrow > qg);
          // dS = P (dP - delta) scale; Ds holds delta * scale
          float const ds = ex[r] * __builtin_fmaf(s[r], p.scale, -Ds[cur][part + ql]);
          ex[r] = masked ? 0.0f : ds;
        }
        if (SAVE && kv0 < p.Skv) save_scores(p, pair, qt0, kvrow, h32, ex);
      }
      // dV += P^T dO or dK += dS^T Q: A = the accumulator (row = key), B = rows of the
      // matching query, reduction over the tile's queries
      contract_rows<DP / 32, C::kStrideB, false>((role == 0 ? Gs[cur] : Qs[cur]) + (part + 4 * h32) * C::kStrideB + l32, ex, acc);
    }
    if (more) {
      st.land(Qs[cur ^ 1], Gs[cur ^ 1]);
      store_row_terms(cur ^ 1);
    }
    __syncthreads();
    cur ^= 1;
  }

  if constexpr (KW > 1) {
    float *const slot = &Qs[0][0] + role * DP * 32;
    static_assert(2 * DP * 32 <= 2 * T * C::kStrideB, "the sums fit the tiles' room");
    if (blk > 0) acc_put<DP / 32>(slot, acc, lane);
    __syncthreads();
    if (blk > 0) return;
    acc_add<DP / 32>(slot, 1.0f, acc, lane);
  }
  // accumulator element r: key row 8*(r/4) + 4*h + r%4 of this wave's 32, column d = i*32 + l%32
  float *op = role == 0 ? p.dv + (int64_t)b * p.v_bs + (int64_t)head * p.Dv : p.dk + (int64_t)b * p.k_bs + (int64_t)head * p.Dq;
  int64_t const oss = role == 0 ? p.v_ss : p.k_ss;
  int const D = role == 0 ? p.Dv : p.Dq;
#pragma unroll
  for (int i = 0; i < DP / 32; i++) {
    int const d = i * 32 + l32;
#pragma unroll
    for (int r = 0; r < 16; r++) {
      int const grow = kv0 + 8 * (r >> 2) + 4 * h32 + (r & 3);
      if (grow < p.Skv && d < D) op[(int64_t)grow * oss + d] = acc[i][r];
    }
  }
}

// dQ: role 0 computes S and P, role 1 dP; each hands the other its tile, both form dS, and each
// produces half of dQ's columns.
template <int DP, bool DMA, int KW>
__global__ __launch_bounds__(256) void attn_f32_bwd_dq_pair_kernel(AttnF32Params p) {
  using C = AttnF32Cfg<DP>;
  constexpr int T = 32 * KW, QR = 64 / KW;
  __shared__ __attribute__((aligned(16))) float Ks[2][T * C::kStrideB];
  __shared__ __attribute__((aligned(16))) float Vs[2][T * C::kStrideA];
  __shared__ PairTile Xs[2][2];
  int const t = threadIdx.x, lane = t & 63, h32 = lane >> 5, l32 = lane & 31;
  int const wave = __builtin_amdgcn_readfirstlane(t >> 6);
  int const blk = wave & 1, role = wave >> 1;
  int const nqb = (p.Sq + QR - 1) / QR;
  int const hb = blockIdx.x % (p.H * p.B);
  int const qb = nqb - 1 - blockIdx.x / (p.H * p.B);
  int const head = hb % p.H, b = hb / p.H;
  int const q0 = qb * QR + (KW == 1 ? blk * 32 : 0);  // this wave's first query
  int const part = KW == 1 ? 0 : blk * 32;             // its first key of a step
  int const qrow = q0 + l32;
  int const rq = min(qrow, p.Sq - 1);
  float own[DP / 2];  // role 0: the row of Q, role 1: of dO
  if (role == 0) load_owned_row<DP>(p.q + (int64_t)b * p.q_bs + (int64_t)head * p.Dq + (int64_t)rq * p.q_ss, p.Dq, h32, own);
  else load_owned_row<DP>(p.d_o + (int64_t)b * p.o_bs + (int64_t)head * p.Dv + (int64_t)rq * p.o_ss, p.Dv, h32, own);
  float const lse2 = p.lse[((int64_t)b * p.H + head) * p.Sq + rq] * kLog2eF;
  float const delta_s = p.delta[((int64_t)b * p.H + head) * p.Sq + rq] * p.scale;
  f32x16 dq[DP / 64];
#pragma unroll
  for (int i = 0; i < DP / 64; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) dq[i][r] = 0.0f;

  int kv_end = p.Skv;
  if (p.causal) kv_end = min(p.Skv, qb * QR + QR);
  int const ntiles = (kv_end + T - 1) / T;
  PairStream<DP, DMA, C::kStrideB, C::kStrideA, T> st;
  st.base[0] = p.k + (int64_t)b * p.k_bs + (int64_t)head * p.Dq;
  st.base[1] = p.v + (int64_t)b * p.v_bs + (int64_t)head * p.Dv;
  st.ss[0] = p.k_ss; st.ss[1] = p.v_ss;
  st.D[0] = p.Dq; st.D[1] = p.Dv;
  st.last = p.Skv - 1; st.t = t; st.lane = lane; st.wave = wave;
  st.init();
  st.fetch(0, Ks[0], Vs[0]);
  st.land(Ks[0], Vs[0]);
  if constexpr (DMA) wait_all_vmem_known_to_compiler();
  __syncthreads();
  int cur = 0;
  for (int it = 0; it < ntiles; it++) {
    int const kt0 = it * T + part;
    bool const more = it + 1 < ntiles;
    if (more) st.fetch((it + 1) * T, Ks[cur ^ 1], Vs[cur ^ 1]);
    bool const active = (KW == 1 || kt0 < p.Skv) && (!p.causal || kt0 <= q0 + 31);
    float ex[16];  // role 0: P, role 1: (dP - delta) scale
    if (active) {
      // S^T = K Q^T or dP^T = V dO^T: rows = keys of the tile, column = this lane's query
      f32x16 s;
#pragma unroll
      for (int r = 0; r < 16; r++) s[r] = 0.0f;
      contract_d<DP>(role == 0 ? Ks[cur] + (part + l32) * C::kStrideB + h32 * (DP / 2) : Vs[cur] + (part + l32) * C::kStrideA + h32 * (DP / 2),
                     own, s);
#pragma unroll
      for (int r = 0; r < 16; r++) {
        int const kv = kt0 + 8 * (r >> 2) + 4 * h32 + (r & 3);
        bool const masked = kv >= p.Skv || (p.causal && kv > qrow);
        // both sides of a masked product are 0
        ex[r] = masked ? 0.0f
                       : (role == 0 ? __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], p.scale_log2, -lse2))
                                    : __builtin_fmaf(s[r], p.scale, -delta_s));
      }
      pair_put(Xs[blk][role], lane, ex);
    }
    pair_barrier();
    if (active) {
      float other[16];
      pair_get(Xs[blk][role ^ 1], lane, other);
#pragma unroll
      for (int r = 0; r < 16; r++) ex[r] *= other[r];
      // dQ^T += K^T dS^T: A = K^T (row d), B = dS^T, reduction over the tile's keys
      contract_rows<DP / 64, C::kStrideB, true>(Ks[cur] + (part + 4 * h32) * C::kStrideB + role * (DP / 2) + l32, ex, dq);
    }
    if (more) st.land(Ks[cur ^ 1], Vs[cur ^ 1]);
    __syncthreads();
    cur ^= 1;
  }

  if constexpr (KW > 1) {
    float *const slot = &Ks[0][0] + role * (DP / 2) * 32;
    if (blk > 0) acc_put<DP / 64>(slot, dq, lane);
    __syncthreads();
    if (blk > 0) return;
    acc_add<DP / 64>(slot, 1.0f, dq, lane);
  }
  if (qrow < p.Sq) {
    float *dqp = p.dq + (int64_t)b * p.q_bs + (int64_t)qrow * p.q_ss + (int64_t)head * p.Dq;
#pragma unroll
    for (int i = 0; i < DP / 64; i++) {
#pragma unroll
      for (int g = 0; g < 4; g++) {
        int const d = role * (DP / 2) + i * 32 + 8 * g + 4 * h32;
        if (d < p.Dq) {
          f32x4 w = {dq[i][4 * g], dq[i][4 * g + 1], dq[i][4 * g + 2], dq[i][4 * g + 3]};
          *reinterpret_cast<f32x4 *>(dqp + d) = w;
        }
      }
    }
  }
}

// dQ from the dS that dK and dV's kernel has left: one product instead of the three that it takes to compute
// dS again.  A workgroup's four waves own groups of 32 query rows, CW of them share a group and take DP / CW
// columns each; the waves read dS from memory in the layout of an operand, a tile ahead, and K's tiles from LDS.
// Bound by the fp32 matrix pipe: batch 8 x 8 heads x 512 at head size 256 274 -> 87 us, 98 TFLOP/s, while the stores of
// dS (67 MB) lengthen dK and dV's kernel from 351 to 364; 4 x 8 heads x 508 at 64, whole block, 319 -> 296; no size
// measured, down to 37 rows, got slower.  The products are added up in the order of a kernel whose waves
// do not share out the keys, to the same bits.
template <int DP, bool DMA, int CW>
__global__ __launch_bounds__(256) void attn_f32_bwd_dq_from_scores_kernel(AttnF32Params p) {
  using C = AttnF32Cfg<DP>;
  constexpr int ROWS = 128 / CW, T = C::kTile, N = DP / 32 / CW;
  __shared__ __attribute__((aligned(16))) float Ks[2][T * C::kStrideB];
  int const t = threadIdx.x, lane = t & 63, h32 = lane >> 5, l32 = lane & 31;
  int const wave = __builtin_amdgcn_readfirstlane(t >> 6);
  int const blk = wave % (4 / CW), part = wave / (4 / CW);
  int const nqb = (p.Sq + ROWS - 1) / ROWS;
  int const pair = blockIdx.x % p.pairs, hb = p.pair0 + pair;
  int const qb = nqb - 1 - blockIdx.x / p.pairs;  // heaviest causal blocks first
  int const head = hb % p.H, b = hb / p.H;
  int const q0 = qb * ROWS + blk * 32, qrow = q0 + l32;
  float const *kp = p.k + (int64_t)b * p.k_bs + (int64_t)head * p.Dq;
  float const *const scores = p.ds + ((int64_t)pair * p.Sq + min(qrow, p.Sq - 1)) * p.ds_ld + 4 * h32;
  f32x16 dq[N];
#pragma unroll
  for (int i = 0; i < N; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) dq[i][r] = 0.0f;

  int kv_end = p.Skv;
  if (p.causal) kv_end = min(p.Skv, qb * ROWS + ROWS);
  int const ntiles = (kv_end + T - 1) / T;
  // the tiles that this wave's rows see, and that dK and dV's kernel has written: keys up to the rows' own
  int const mine = p.causal ? min(ntiles, q0 / T + 1) : ntiles;
  f32x4 rk[C::kChunks], next[4];
  i32x4 rsrc;
  unsigned lane_off = 0;
  if constexpr (DMA) {
    rsrc = buffer_resource(kp, kRowsBound);
    lane_off = row_lane_offset(lane, p.Dq);
  }
  auto fetch = [&](int it, int buf) __attribute__((always_inline)) {
    if constexpr (DMA) tile_dma<C::kStrideB>(rsrc, lane_off, p.k_ss, it * T, p.Skv - 1, wave, Ks[buf]);
    else tile_gload<DP>(kp, p.k_ss, it * T, p.Skv - 1, p.Dq, t, rk);
    if (it < mine) {
#pragma unroll
      for (int g = 0; g < 4; g++) next[g] = *reinterpret_cast<f32x4 const *>(scores + it * T + 8 * g);
    }
  };
  float ds[16];
  auto land = [&](int buf) __attribute__((always_inline)) {
    if constexpr (DMA) wait_vmcnt<0>();
    else tile_lstore<DP, C::kStrideB>(Ks[buf], t, rk);
#pragma unroll
    for (int g = 0; g < 4; g++)
#pragma unroll
      for (int e = 0; e < 4; e++) ds[4 * g + e] = next[g][e];
  };
#pragma unroll
  for (int g = 0; g < 4; g++) next[g] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  fetch(0, 0);
  land(0);
  if constexpr (DMA) wait_all_vmem_known_to_compiler();
  __syncthreads();
  int cur = 0;
  for (int it = 0; it < ntiles; it++) {
    bool const more = it + 1 < ntiles;
    if (more) fetch(it + 1, cur ^ 1);
    // dQ^T += K^T dS^T: A = K^T (row d), B = dS^T, reduction over the tile's keys
    if (it < mine) contract_rows<N, C::kStrideB, true>(Ks[cur] + 4 * h32 * C::kStrideB + part * (DP / CW) + l32, ds, dq);
    if (more) land(cur ^ 1);
    __syncthreads();
    cur ^= 1;
  }
  if (qrow < p.Sq) {
    float *dqp = p.dq + (int64_t)b * p.q_bs + (int64_t)qrow * p.q_ss + (int64_t)head * p.Dq;
#pragma unroll
    for (int i = 0; i < N; i++) {
#pragma unroll
      for (int g = 0; g < 4; g++) {
        int const d = part * (DP / CW) + i * 32 + 8 * g + 4 * h32;
        if (d < p.Dq) *reinterpret_cast<f32x4 *>(dqp + d) = f32x4{dq[i][4 * g], dq[i][4 * g + 1], dq[i][4 * g + 2], dq[i][4 * g + 3]};
      }
    }
  }
}

static int check_desc_f32(char const *who, ffk_attention_desc_t const *d) {
  int64_t const dq = d->head_dim, dv = d->v_head_dim > 0 ? d->v_head_dim : d->head_dim;
  FFK_REQUIRE(dq > 0 && dq <= 256 && dq % 4 == 0 && dv <= 256 && dv % 4 == 0,
              "%s: fp32 head_dim %lld / v_head_dim %lld not supported (multiples of 4 up to 256)", who,
              (long long)dq, (long long)dv);
  FFK_REQUIRE(d->batch > 0 && d->heads > 0 && d->seq_q > 0 && d->seq_kv > 0, "%s: bad shape", who);
  FFK_REQUIRE(d->batch * d->heads * ((d->seq_q > d->seq_kv ? d->seq_q : d->seq_kv) / 64 + 1) < (1ll << 32),
              "%s: too many workgroups", who);
  FFK_REQUIRE(d->seq_q < (1ll << 30) && d->seq_kv < (1ll << 30), "%s: sequence too long", who);
  FFK_REQUIRE(d->q_seq_stride % 4 == 0 && d->k_seq_stride % 4 == 0 && d->v_seq_stride % 4 == 0 &&
                  d->o_seq_stride % 4 == 0 && d->q_batch_stride % 4 == 0 && d->k_batch_stride % 4 == 0 &&
                  d->v_batch_stride % 4 == 0 && d->o_batch_stride % 4 == 0,
              "%s: fp32 strides must be multiples of 4 elements", who);
  FFK_REQUIRE(d->q_seq_stride >= d->heads * dq && d->k_seq_stride >= d->heads * dq &&
                  d->v_seq_stride >= d->heads * dv && d->o_seq_stride >= d->heads * dv,
              "%s: sequence stride smaller than heads * head_dim", who);
  return FFK_OK;
}

static AttnF32Params make_params(ffk_attention_desc_t const *d) {
  AttnF32Params p = {};
  p.B = (int)d->batch; p.H = (int)d->heads; p.Sq = (int)d->seq_q; p.Skv = (int)d->seq_kv;
  p.Dq = (int)d->head_dim;
  p.Dv = (int)(d->v_head_dim > 0 ? d->v_head_dim : d->head_dim);
  p.q_bs = d->q_batch_stride; p.q_ss = d->q_seq_stride;
  p.k_bs = d->k_batch_stride; p.k_ss = d->k_seq_stride;
  p.v_bs = d->v_batch_stride; p.v_ss = d->v_seq_stride;
  p.o_bs = d->o_batch_stride; p.o_ss = d->o_seq_stride;
  p.scale = d->scale;
  p.scale_log2 = d->scale * kLog2eF;
  p.causal = d->causal;
  p.pairs = p.B * p.H;
  return p;
}

// Rows of every operand within 31 bits of their (batch, head)'s first element: direct loads reach them.
static bool rows_fit_dma(AttnF32Params const &p) {
  auto fits = [](int64_t rows, int64_t stride) { return stride < (1 << 28) && rows * stride * 4 < (int64_t)kRowsBound; };
  return fits(p.Sq, p.q_ss) && fits(p.Skv, p.k_ss) && fits(p.Skv, p.v_ss) && fits(p.Sq, p.o_ss);
}

#define FFK_ATTN_F32_DISPATCH(D_, CALL)                                        \
  do {                                                                         \
    if ((D_) <= 32) { CALL(32, false); }                                       \
    else if ((D_) <= 64) { CALL(64, false); }                                  \
    else if ((D_) <= 128) { CALL(128, false); }                                \
    else if (rows_fit_dma(p)) { CALL(256, true); }                             \
    else { CALL(256, false); }                                                 \
  } while (0)

// How many waves, or pairs of them, share a group's rows: as many as leave one round of workgroups, two under a causal
// mask, where half of them are short.  In us by 1, 2, 4 ([B, S, D] x heads; forward, dK and dV by 1, 2):
//   [3, 305, 128] x 4   60 38 31, 63 38      [5, 219, 64] x 4, causal   27 19 15, 29 20
//   [5, 215, 128] x 8   45 33 42, 46 60      [2, 600, 128] x 8, causal  101 64 44, 111 69
//   [2, 376, 64] x 16   44 29 34, 49 55      [5, 609, 128] x 8, causal  111 70 94, 124 131
static int f32_split(AttnF32Params const &p, int rows_owned, int rows, int streamed, int most) {
  int64_t const heads = (int64_t)p.H * p.B, limit = p.causal ? 2 * kNumCU : kNumCU;
  int kw = 1;
  while (kw < most && heads * ceil_div(rows_owned, rows / (2 * kw)) <= limit && streamed > 32 * kw) kw *= 2;
  return kw;
}

template <int DP, bool DMA>
static void launch_f32_forward(hipStream_t st, AttnF32Params const &p) {
  int const kw = DP <= 128 ? f32_split(p, p.Sq, 128, p.Skv, 4) : 1;
  unsigned const grid = (unsigned)(ceil_div(p.Sq, 128 / kw) * p.H * p.B);
  if constexpr (DP <= 128) {
    if (kw == 4) return (void)(attn_f32_fwd_kernel<DP, DMA, 4><<<grid, 256, 0, st>>>(p));
    if (kw == 2) return (void)(attn_f32_fwd_kernel<DP, DMA, 2><<<grid, 256, 0, st>>>(p));
  }
  attn_f32_fwd_kernel<DP, DMA, 1><<<grid, 256, 0, st>>>(p);
}

int attention_f32_forward(hipStream_t st, ffk_attention_desc_t const *d, void const *q, void const *k,
                          void const *v, void *o, float *lse) {
  int rc = check_desc_f32("attention_forward", d);
  if (rc != FFK_OK) return rc;
  AttnF32Params p = make_params(d);
  p.q = static_cast<float const *>(q);
  p.k = static_cast<float const *>(k);
  p.v = static_cast<float const *>(v);
  p.out = static_cast<float *>(o);
  p.lse = lse;
  int const dmax = p.Dq > p.Dv ? p.Dq : p.Dv;
#define CALL(DP_, DMA_) launch_f32_forward<DP_, DMA_>(st, p)
  FFK_ATTN_F32_DISPATCH(dmax, CALL);
#undef CALL
  FFK_CHECK_LAUNCH();
  return FFK_OK;
}

// Scratch for dS, which lets dQ's kernel skip two of its three products: how many pairs of batch entry and head go into
// `bytes` of it at a time, all of them, or as many in several launches where those still fill the chip twice over; 0: no use
// of it.  Half a GB holds dS of every block of up to 700 rows that was measured; where it does not, a launch for a
// part of the heads still has two workgroups a CU.  What is asked for is what is used: by this rule too.
constexpr size_t kMostScores = (size_t)512 << 20;
static int64_t f32_scores_row(int64_t seq_kv) { return ceil_div(seq_kv, 32) * 32; }
static int64_t f32_pairs_at_a_time(int64_t pairs, int64_t seq_q, int64_t seq_kv, size_t bytes) {
  if (pairs <= 0 || seq_q <= 0 || seq_kv <= 0 || seq_q >= (1 << 30) || seq_kv >= (1 << 30)) return 0;
  if ((seq_q + 96) * f32_scores_row(seq_kv) * (int64_t)sizeof(float) > (int64_t)1 << 32) return 0;  // 32-bit offsets (save_scores)
  int64_t const most = (int64_t)(std::min(bytes, kMostScores) / ((size_t)seq_q * f32_scores_row(seq_kv) * sizeof(float)));
  if (most >= pairs) return pairs;
  return most * ceil_div(std::min(seq_q, seq_kv), 128) >= 2 * kNumCU ? most : 0;
}
size_t attention_f32_scores_bytes(int64_t pairs, int64_t seq_q, int64_t seq_kv) {
  return (size_t)f32_pairs_at_a_time(pairs, seq_q, seq_kv, kMostScores) * (size_t)seq_q * f32_scores_row(seq_kv) * sizeof(float);
}

template <int DP, bool DMA>
static void launch_f32_backward(hipStream_t st, AttnF32Params const &p, int64_t rows, void *scratch, size_t scratch_bytes) {
  attn_f32_delta_kernel<DP><<<(unsigned)ceil_div(rows, 4 * (64 / (DP / 4))), 256, 0, st>>>(p);
  int64_t const heads = (int64_t)p.H * p.B;
  // Pairs always at 256 (see above) and at 64, where they leave registers for twice the waves (batch 6 x 32
  // heads x 700, causal: dK/dV 358 -> 297 us, dQ 235 -> 212); at 128 while workgroups of 128 rows do not fill
  // the chip (8 heads, 138 x 58, head size 80: dK/dV 56 -> 35 us; 2 x 32 heads x 469: 173 -> 196, so not there).
  auto pairs = [&](int64_t rows_owned) {
    return DP >= 64 && (DP != 128 || ceil_div(rows_owned, 128) * heads < kNumCU);
  };
  auto launch_dkdv = [&](AttnF32Params const &q, auto save) {
    constexpr bool SAVE = decltype(save)::value;
    int64_t const n = q.pairs;
    if constexpr (DP >= 64) {
      if (pairs(p.Skv)) {
        int const kw = f32_split(p, p.Skv, 64, p.Sq, DP <= 128 ? 2 : 1);
        if constexpr (DP <= 128) {
          if (kw == 2) return (void)(attn_f32_bwd_dkdv_pair_kernel<DP, DMA, 2, SAVE><<<(unsigned)(ceil_div(p.Skv, 32) * n), 256, 0, st>>>(q));
        }
        attn_f32_bwd_dkdv_pair_kernel<DP, DMA, 1, SAVE><<<(unsigned)(ceil_div(p.Skv, 64) * n), 256, 0, st>>>(q);
        return;
      }
    }
    if constexpr (DP == 32 || DP == 128) {
      attn_f32_bwd_dkdv_kernel<DP, SAVE><<<(unsigned)(ceil_div(p.Skv, 128) * n), 256, 0, st>>>(q);
    }
  };
  if (int64_t const at_a_time = f32_pairs_at_a_time(heads, p.Sq, p.Skv, scratch_bytes); scratch != nullptr && at_a_time > 0) {
    AttnF32Params q = p;
    q.ds = static_cast<float *>(scratch);
    q.ds_ld = (int)f32_scores_row(p.Skv);
    for (q.pair0 = 0; q.pair0 < heads; q.pair0 += q.pairs) {
      q.pairs = (int)std::min<int64_t>(at_a_time, heads - q.pair0);
      launch_dkdv(q, std::true_type{});
      // few columns a wave where so many rows a workgroup leave CUs without one (3 x 4 heads x 633 of 64, causal, whole
      // block: 183 us by the kernel that computes dS again, 186 with 128 rows a workgroup, 176 with 64)
      constexpr int CW = DP <= 64 ? 1 : 2, MORE = DP >= 64 ? 2 * CW : CW;
      if (MORE > CW && ceil_div(p.Sq, 128 / CW) * q.pairs < kNumCU) {
        attn_f32_bwd_dq_from_scores_kernel<DP, DMA, MORE><<<(unsigned)(ceil_div(p.Sq, 128 / MORE) * q.pairs), 256, 0, st>>>(q);
      } else {
        attn_f32_bwd_dq_from_scores_kernel<DP, DMA, CW><<<(unsigned)(ceil_div(p.Sq, 128 / CW) * q.pairs), 256, 0, st>>>(q);
      }
    }
    return;
  }
  launch_dkdv(p, std::false_type{});
  if constexpr (DP >= 64) {
    if (pairs(p.Sq)) {
      int const kw = f32_split(p, p.Sq, 64, p.Skv, DP <= 128 ? 2 : 1);
      if constexpr (DP <= 128) {
        if (kw == 2) return (void)(attn_f32_bwd_dq_pair_kernel<DP, DMA, 2><<<(unsigned)(ceil_div(p.Sq, 32) * heads), 256, 0, st>>>(p));
      }
      attn_f32_bwd_dq_pair_kernel<DP, DMA, 1><<<(unsigned)(ceil_div(p.Sq, 64) * heads), 256, 0, st>>>(p);
      return;
    }
  }
  if constexpr (DP == 32 || DP == 128) attn_f32_bwd_dq_kernel<DP><<<(unsigned)(ceil_div(p.Sq, 128) * heads), 256, 0, st>>>(p);
}

int attention_f32_backward(hipStream_t st, ffk_attention_desc_t const *d, void const *q, void const *k,
                           void const *v, void const *o, void const *d_o, float const *lse, float *delta,
                           void *dq, void *dk, void *dv, void *scratch, size_t scratch_bytes) {
  int rc = check_desc_f32("attention_backward", d);
  if (rc != FFK_OK) return rc;
  AttnF32Params p = make_params(d);
  p.q = static_cast<float const *>(q);
  p.k = static_cast<float const *>(k);
  p.v = static_cast<float const *>(v);
  p.o = static_cast<float const *>(o);
  p.d_o = static_cast<float const *>(d_o);
  p.lse = const_cast<float *>(lse);
  p.delta = delta;
  p.dq = static_cast<float *>(dq);
  p.dk = static_cast<float *>(dk);
  p.dv = static_cast<float *>(dv);
  int64_t const rows = (int64_t)p.B * p.H * p.Sq;
  int const dmax = p.Dq > p.Dv ? p.Dq : p.Dv;
#define CALL(DP_, DMA_) launch_f32_backward<DP_, DMA_>(st, p, rows, scratch, scratch_bytes)
  FFK_ATTN_F32_DISPATCH(dmax, CALL);
#undef CALL
  FFK_CHECK_LAUNCH();
  return FFK_OK;
}

}  // namespace ffk
