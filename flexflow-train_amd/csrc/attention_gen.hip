// Fused attention for gfx950, bf16 operands / fp32 accumulation, for the head
// sizes the tuned kernels of attention.hip do not take: any multiple of 8 up to
// 256, and a value head size (V, O, dO, dV) that differs from the query/key one
// (Q, K, dQ, dK).  The reference's model builders ask for kdim = vdim = 256
// (lib/models/src/models/transformer/transformer.cc:37-38, bert/bert.cc:64-65)
// and its attributes leave the two projection sizes free
// (lib/op-attrs/src/op-attrs/ops/attention.cc:23-37).
//
// Same scheme as attention.hip (scores computed transposed so a lane owns one
// query's column, probabilities fed to the next product from registers, the
// backward as two kernels without atomics): DP is the larger head size rounded up to
// 32, 64, 96, 128 or 256, columns past a tensor's own head size are zeros in LDS and
// never stored; tiles travel global -> registers -> LDS one step ahead.
//   The four waves of a workgroup are 4 / KW groups of 32 rows, and the KW waves of a group take the streamed
// rows in turn; what they accumulated meets in LDS at the end.  KW > 1 is for problems that would leave CUs
// without a workgroup: more of them, each with fewer steps.
#include "attention_common.h"

namespace ffk {

struct AttnGenParams {
  bf16 const *q, *k, *v, *o, *d_o;
  bf16 *out;
  float *lse;    // forward: written; backward: read
  float *delta;  // backward: written by the dQ kernel, read by the dK/dV kernel
  bf16 *dq, *dk, *dv;
  int B, H, Sq, Skv, Dq, Dv;
  int64_t q_bs, q_ss, k_bs, k_ss, v_bs, v_ss, o_bs, o_ss;
  float scale, scale_log2;
  int causal;
};

// Row strides of LDS tiles, in elements, free of bank conflicts for 16-byte reads of 16 rows (row), for
// transposing reads of 4 rows x 64 bytes (turned), or nearly so for both.
template <int DP>
struct GenStride {
  static constexpr int row = DP + 8;
  static constexpr int turned = DP == 32 || DP == 96 ? DP : DP + 32;
  static constexpr int both = DP == 32 ? 40 : DP == 96 ? 104 : DP + 40;
};
constexpr int kGenLds = 80 * 1024;
__device__ __forceinline__ u32x4 load8_or_zero(bf16 const *row, int d0, int D) {
  u32x4 z = {0u, 0u, 0u, 0u};
  return d0 < D ? *reinterpret_cast<u32x4 const *>(row + d0) : z;
}

// This lane's row of an owned operand as B-operand fragments (column = the row, k = d).
template <int DP>
__device__ __forceinline__ void gen_load_owned(bf16 const *row, int D, int h32, bf16x8 (&f)[DP / 16]) {
#pragma unroll
  for (int kk = 0; kk < DP / 16; kk++) {
    union {
      u32x4 u;
      bf16x8 b;
    } x;
    x.u = load8_or_zero(row, kk * 16 + h32 * 8, D);
    f[kk] = x.b;
  }
}

// A tile of T rows on its way from memory to LDS (rows past the last one repeat it).  Columns past the
// tensor's own head size are cleared once in every buffer and not written again.
template <int DP, int T>
struct GenTile {
  static constexpr int kCPR = DP == 96 ? 16 : DP / 8;  // 16-byte chunks a row has threads for
  static constexpr int kRows = 256 / kCPR, kN = (T + kRows - 1) / kRows;
  u32x4 r[kN];
  __device__ __forceinline__ void load(bf16 const *base, int64_t row_stride, int row0, int last_row, int D, int t) {
    int const col = min((t % kCPR) * 8, D - 8);
#pragma unroll
    for (int i = 0; i < kN; i++) {
      int const gr = min(row0 + t / kCPR + i * kRows, last_row);
      r[i] = *reinterpret_cast<u32x4 const *>(base + (int64_t)gr * row_stride + col);
    }
  }
  __device__ __forceinline__ void store(bf16 *tile, int stride, int D, int t) const {
    int const ch = t % kCPR;
    if (ch * 8 < D) {
#pragma unroll
      for (int i = 0; i < kN; i++) {
        int const row = t / kCPR + i * kRows;
        if (T >= kRows || row < T) *reinterpret_cast<u32x4 *>(tile + row * stride + ch * 8) = r[i];
      }
    }
  }
  __device__ __forceinline__ static void clear(bf16 *tile, int stride, int D, int t) {
    int const ch = t % kCPR;
    if (ch * 8 >= D && ch * 8 < DP) {
#pragma unroll
      for (int i = 0; i < kN; i++) {
        int const row = t / kCPR + i * kRows;
        if (T >= kRows || row < T) *reinterpret_cast<u32x4 *>(tile + row * stride + ch * 8) = u32x4{0u, 0u, 0u, 0u};
      }
    }
  }
};

// A wave's accumulators to LDS and back, for the wave that adds them up: 16 bytes a lane, lanes side by side.
template <int NI>
__device__ __forceinline__ void gen_put(float *to, f32x16 const (&acc)[NI], int lane) {
#pragma unroll
  for (int i = 0; i < NI; i++)
#pragma unroll
    for (int g = 0; g < 4; g++)
      *reinterpret_cast<f32x4 *>(to + ((i * 4 + g) * 64 + lane) * 4) =
          f32x4{acc[i][4 * g], acc[i][4 * g + 1], acc[i][4 * g + 2], acc[i][4 * g + 3]};
}
template <int NI>
__device__ __forceinline__ void gen_add(float const *from, float factor, f32x16 (&acc)[NI], int lane) {
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
// forward: workgroup = 128 / KW query rows of one (batch, head)
// --------------------------------------------------------------------------
template <int DP, int KW>
struct GenFwd {
  static constexpr int kJ = DP <= 128 && KW <= 2 ? 2 : 1;  // 32-key blocks of a wave and step
  static constexpr int kT = 32 * kJ * KW;
  static constexpr int kTile = kT * (GenStride<DP>::row + GenStride<DP>::turned);  // elements, K and V
  static constexpr int kBuffers = 2 * kTile * 2 <= kGenLds ? 2 : 1;
  static constexpr int kMerge = (KW - 1) * (4 / KW) * (DP * 32 + 128) * 4;  // bytes
  static constexpr int kBytes = kBuffers * kTile * 2 > kMerge ? kBuffers * kTile * 2 : kMerge;
};
template <int DP, int KW>
__global__ __launch_bounds__(256) void attn_gen_fwd_kernel(AttnGenParams p) {
  using C = GenFwd<DP, KW>;
  constexpr int KS = GenStride<DP>::row, VS = GenStride<DP>::turned, J = C::kJ, QR = 128 / KW;
  constexpr int NB = KW * J;  // 32-key blocks of a step
  __shared__ __attribute__((aligned(16))) uint8_t pool[C::kBytes];
  __shared__ float block_max[KW > 1 ? 4 / KW : 1][KW > 1 ? NB : 1][32];
  int const t = threadIdx.x, lane = t & 63, h32 = lane >> 5;
  int const wave = __builtin_amdgcn_readfirstlane(t >> 6);
  int const qw = wave / KW, kw = wave % KW;
  int const nqb = (p.Sq + QR - 1) / QR;
  int const hb = blockIdx.x % (p.H * p.B);
  int const qb = nqb - 1 - blockIdx.x / (p.H * p.B);  // heaviest causal blocks first
  int const head = hb % p.H, b = hb / p.H;
  int const q0 = qb * QR, qw0 = q0 + qw * 32;
  int const qrow = qw0 + (lane & 31);
  bool const in_pairs = p.Dq == p.Dv && (p.Dq == 64 || p.Dq == 128);
  bf16 const *qp = p.q + (int64_t)b * p.q_bs + (int64_t)head * p.Dq;
  bf16 const *kp = p.k + (int64_t)b * p.k_bs + (int64_t)head * p.Dq;
  bf16 const *vp = p.v + (int64_t)b * p.v_bs + (int64_t)head * p.Dv;
  auto k_tile = [&](int buf) { return reinterpret_cast<bf16 *>(pool) + buf * C::kTile; };
  auto v_tile = [&](int buf) { return k_tile(buf) + C::kT * KS; };

  bf16x8 qf[DP / 16];
  gen_load_owned<DP>(qp + (int64_t)min(qrow, p.Sq - 1) * p.q_ss, p.Dq, h32, qf);

  int kv_end = p.Skv;
  if (p.causal) kv_end = min(p.Skv, q0 + QR);
  int const ntiles = (kv_end + C::kT - 1) / C::kT;

  f32x16 oacc[DP / 32];
#pragma unroll
  for (int i = 0; i < DP / 32; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) oacc[i][r] = 0.0f;
  float m_run = -INFINITY, m_own = -INFINITY, l_run = 0.0f;  // largest score of all waves' keys, what P is relative to

  GenTile<DP, C::kT> tk, tv;
  auto fetch = [&](int kv0) {
    tk.load(kp, p.k_ss, kv0, p.Skv - 1, p.Dq, t);
    tv.load(vp, p.v_ss, kv0, p.Skv - 1, p.Dv, t);
  };
  auto stash = [&](int buf) {
    tk.store(k_tile(buf), KS, p.Dq, t);
    tv.store(v_tile(buf), VS, p.Dv, t);
  };
  int const koff = lane_k_off(KS, lane);
  int const toff = lane_tr_off(VS, lane);
  fetch(0);
#pragma unroll
  for (int buf = 0; buf < C::kBuffers; buf++) {
    GenTile<DP, C::kT>::clear(k_tile(buf), KS, p.Dq, t);
    GenTile<DP, C::kT>::clear(v_tile(buf), VS, p.Dv, t);
  }
  stash(0);
  __syncthreads();
  int cur = 0;
  for (int it = 0; it < ntiles; it++) {
    bool const more = it + 1 < ntiles;
    if (more) fetch((it + 1) * C::kT);
    int const kv0 = it * C::kT + kw * 32 * J;  // this wave's keys
    // a wave whose rows all lie before its keys (causal), or whose keys do not exist, has nothing to add
    bool const active = kv0 < p.Skv && (!p.causal || kv0 <= qw0 + 31);
    // S^T: rows = keys, column = this lane's query; the largest score of each block of 32 keys
    f32x16 s[J];
    float mx[J];
#pragma unroll
    for (int j = 0; j < J; j++) mx[j] = -INFINITY;
    if (active) {
      bf16 const *kt = k_tile(cur) + kw * 32 * J * KS + koff;
#pragma unroll
      for (int j = 0; j < J; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) s[j][r] = 0.0f;
#pragma unroll
      for (int kk = 0; kk < DP / 16; kk++)
#pragma unroll
        for (int j = 0; j < J; j++) {
          bf16x8 const kf = frag_k(kt, KS, j * 32, kk * 16);
          s[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[kk], s[j], 0, 0, 0);
        }
      bool const need_mask = (kv0 + 32 * J > p.Skv) || (p.causal && kv0 + 32 * J - 1 > qw0);
      if (need_mask) {
#pragma unroll
        for (int j = 0; j < J; j++)
#pragma unroll
          for (int r = 0; r < 16; r++) {
            int const kv = kv0 + j * 32 + 8 * (r >> 2) + 4 * h32 + (r & 3);
            if (kv >= p.Skv || (p.causal && kv > qrow)) s[j][r] = -INFINITY;
          }
      }
#pragma unroll
      for (int j = 0; j < J; j++) {
#pragma unroll
        for (int r = 0; r < 16; r++) mx[j] = fmaxf(mx[j], s[j][r]);
        mx[j] = max_across_halves(mx[j]) * p.scale_log2;
      }
    }
    // What P is relative to: the largest score up to its block's end, also of the other waves' blocks, as if one wave
    // walked them all, blocks of 64 keys at the head sizes of the kernels that step by 64.  P is rounded to bf16, so
    // with another maximum each of its roundings falls differently, and results of two splits of the rows would be
    // apart by 1e-3; so they differ in the order of fp32 sums alone (one barrier a step; [2, 1198] x 4 heads of 64, 80
    // workgroups 22 us, 18.7 with a maximum for each wave, 23.7 without shares).  Finite: key 0 is visible to every
    // query.
    float m_block[J], m_step = m_run;
    if constexpr (KW > 1) {
      if (lane < 32) {
#pragma unroll
        for (int j = 0; j < J; j++) block_max[qw][kw * J + j][lane] = mx[j];
      }
      __syncthreads();
#pragma unroll
      for (int n = 0; n < NB; n++) {
        float const now = block_max[qw][n][lane & 31];
        float const ahead = n % 2 == 0 && in_pairs ? fmaxf(now, block_max[qw][n + 1][lane & 31]) : now;
        m_step = fmaxf(m_step, ahead);
#pragma unroll
        for (int j = 0; j < J; j++)
          if (n == kw * J + j) m_block[j] = m_step;
      }
    } else {
#pragma unroll
      for (int j = 0; j < J; j++) {
        m_step = fmaxf(m_step, j % 2 == 0 && J > 1 && in_pairs ? fmaxf(mx[j], mx[J - 1]) : mx[j]);
        m_block[j] = m_step;
      }
    }
    m_run = m_step;
    if (active) {
      bf16 const *vt = v_tile(cur) + kw * 32 * J * VS + toff;
      float alpha[J];
      bf16x8 pf[2 * J];
#pragma unroll
      for (int j = 0; j < J; j++) {
        alpha[j] = __builtin_amdgcn_exp2f(m_own - m_block[j]);
        m_own = m_block[j];
        float sum = 0.0f, pv[16];
#pragma unroll
        for (int r = 0; r < 16; r++) {
          pv[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[j][r], p.scale_log2, -m_own));
          sum += pv[r];
        }
        pf[2 * j] = pack8(pv);
        pf[2 * j + 1] = pack8(pv + 8);
        l_run = l_run * alpha[j] + sum;  // this lane's 16 of every 32 keys; the lane halves meet at the end
      }
#pragma unroll
      for (int j = 0; j < J; j++) {
        if (__builtin_amdgcn_ballot_w64(alpha[j] != 1.0f) != 0) {
#pragma unroll
          for (int i = 0; i < DP / 32; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) oacc[i][r] *= alpha[j];
        }
        // O^T += V^T P^T: A = V^T (rows d) through transposing loads, B = P^T
#pragma unroll
        for (int s2 = 0; s2 < 2; s2++)
#pragma unroll
          for (int i = 0; i < DP / 32; i++) {
            bf16x8 const vf = frag_tr_acc(vt, VS, j * 32, s2, i * 32);
            oacc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pf[2 * j + s2], oacc[i], 0, 0, 0);
          }
      }
    }
    if (C::kBuffers == 1) __syncthreads();
    if (more) stash(C::kBuffers == 1 ? 0 : cur ^ 1);
    __syncthreads();
    if (C::kBuffers == 2) cur ^= 1;
  }

  l_run += __shfl_xor(l_run, 32, 64);
  if constexpr (KW > 1) {
    constexpr int kSlot = DP * 32 + 128;
    float *const slots = reinterpret_cast<float *>(pool) + qw * (KW - 1) * kSlot;
    if (kw > 0) {
      float *const mine = slots + (kw - 1) * kSlot;
      gen_put<DP / 32>(mine, oacc, lane);
      mine[DP * 32 + lane] = m_own;
      mine[DP * 32 + 64 + lane] = l_run;
    }
    __syncthreads();
    if (kw > 0) return;
    float const mine = __builtin_amdgcn_exp2f(m_own - m_run);  // (m_run is the same in all of them)
    l_run *= mine;
#pragma unroll
    for (int i = 0; i < DP / 32; i++)
#pragma unroll
      for (int r = 0; r < 16; r++) oacc[i][r] *= mine;
#pragma unroll
    for (int w = 0; w < KW - 1; w++) {
      float const *const other = slots + w * kSlot;
      float const factor = __builtin_amdgcn_exp2f(other[DP * 32 + lane] - m_run);
      l_run += other[DP * 32 + 64 + lane] * factor;
      gen_add<DP / 32>(other, factor, oacc, lane);
    }
  }
  if (qrow < p.Sq) {
    float const inv = 1.0f / l_run;
    bf16 *op = p.out + (int64_t)b * p.o_bs + (int64_t)qrow * p.o_ss + (int64_t)head * p.Dv;
#pragma unroll
    for (int i = 0; i < DP / 32; i++) {
#pragma unroll
      for (int g = 0; g < 4; g++) {
        int const d = i * 32 + 8 * g + 4 * h32;
        if (d < p.Dv) {
          u32x2 w = {pack_bf16x2(oacc[i][4 * g] * inv, oacc[i][4 * g + 1] * inv),
                     pack_bf16x2(oacc[i][4 * g + 2] * inv, oacc[i][4 * g + 3] * inv)};
          *reinterpret_cast<u32x2 *>(op + d) = w;
        }
      }
    }
    if (h32 == 0 && p.lse != nullptr) {
      p.lse[((int64_t)b * p.H + head) * p.Sq + qrow] = (m_run + __log2f(l_run)) * kLn2;
    }
  }
}

// --------------------------------------------------------------------------
// backward (B): dQ, and delta = rowsum(O * dO) for its rows.  Runs first.
// --------------------------------------------------------------------------
template <int DP, int KW>
struct GenDq {
  static constexpr int kJ = DP <= 128 && KW == 1 ? 2 : 1;
  static constexpr int kT = 32 * kJ * KW;
  static constexpr int kTile = kT * (GenStride<DP>::both + GenStride<DP>::row);  // elements, K and V
  static constexpr int kBuffers = 2 * kTile * 2 <= kGenLds ? 2 : 1;
  static constexpr int kMerge = (KW - 1) * (4 / KW) * DP * 32 * 4;  // bytes
  static constexpr int kBytes = kBuffers * kTile * 2 > kMerge ? kBuffers * kTile * 2 : kMerge;
};
template <int DP, int KW>
__global__ __launch_bounds__(256) void attn_gen_bwd_dq_kernel(AttnGenParams p) {
  using C = GenDq<DP, KW>;
  constexpr int KS = GenStride<DP>::both, VS = GenStride<DP>::row, J = C::kJ, QR = 128 / KW;
  __shared__ __attribute__((aligned(16))) uint8_t pool[C::kBytes];
  int const t = threadIdx.x, lane = t & 63, h32 = lane >> 5;
  int const wave = __builtin_amdgcn_readfirstlane(t >> 6);
  int const qw = wave / KW, kw = wave % KW;
  int const nqb = (p.Sq + QR - 1) / QR;
  int const hb = blockIdx.x % (p.H * p.B);
  int const qb = nqb - 1 - blockIdx.x / (p.H * p.B);
  int const head = hb % p.H, b = hb / p.H;
  int const q0 = qb * QR, qw0 = q0 + qw * 32;
  int const qrow = qw0 + (lane & 31);
  bf16 const *qp = p.q + (int64_t)b * p.q_bs + (int64_t)head * p.Dq;
  bf16 const *gp = p.d_o + (int64_t)b * p.o_bs + (int64_t)head * p.Dv;
  bf16 const *op = p.o + (int64_t)b * p.o_bs + (int64_t)head * p.Dv;
  bf16 const *kp = p.k + (int64_t)b * p.k_bs + (int64_t)head * p.Dq;
  bf16 const *vp = p.v + (int64_t)b * p.v_bs + (int64_t)head * p.Dv;
  auto k_tile = [&](int buf) { return reinterpret_cast<bf16 *>(pool) + buf * C::kTile; };
  auto v_tile = [&](int buf) { return k_tile(buf) + C::kT * KS; };

  GenTile<DP, C::kT> tk, tv;
  auto fetch = [&](int kt0) {
    tk.load(kp, p.k_ss, kt0, p.Skv - 1, p.Dq, t);
    tv.load(vp, p.v_ss, kt0, p.Skv - 1, p.Dv, t);
  };
  auto stash = [&](int buf) {
    tk.store(k_tile(buf), KS, p.Dq, t);
    tv.store(v_tile(buf), VS, p.Dv, t);
  };
  fetch(0);
  bf16x8 qf[DP / 16], gf[DP / 16];
  float lse2, delta_s;  // delta_s = delta * scale
  {
    int const r = min(qrow, p.Sq - 1);
    gen_load_owned<DP>(qp + (int64_t)r * p.q_ss, p.Dq, h32, qf);
    gen_load_owned<DP>(gp + (int64_t)r * p.o_ss, p.Dv, h32, gf);
    lse2 = p.lse[((int64_t)b * p.H + head) * p.Sq + r] * kLog2e;
    // delta of this lane's row: the lane holds 8 of every 16 columns, its partner l ^ 32 the rest
    float part = 0.0f;
#pragma unroll
    for (int kk = 0; kk < DP / 16; kk++) {
      union {
        u32x4 u;
        bf16x8 v;
      } of;
      of.u = load8_or_zero(op + (int64_t)r * p.o_ss, kk * 16 + h32 * 8, p.Dv);
#pragma unroll
      for (int e = 0; e < 8; e++) part += (float)of.v[e] * (float)gf[kk][e];
    }
    float const delta = part + __shfl_xor(part, 32, 64);
    if (kw == 0 && h32 == 0 && qrow < p.Sq) p.delta[((int64_t)b * p.H + head) * p.Sq + qrow] = delta;
    delta_s = delta * p.scale;
  }
  f32x16 dq[DP / 32];
#pragma unroll
  for (int i = 0; i < DP / 32; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) dq[i][r] = 0.0f;

  int kv_end = p.Skv;
  if (p.causal) kv_end = min(p.Skv, q0 + QR);
  int const ntiles = (kv_end + C::kT - 1) / C::kT;

  int const koff = lane_k_off(KS, lane), voff = lane_k_off(VS, lane);
  int const toff = lane_tr_off(KS, lane);
#pragma unroll
  for (int buf = 0; buf < C::kBuffers; buf++) {
    GenTile<DP, C::kT>::clear(k_tile(buf), KS, p.Dq, t);
    GenTile<DP, C::kT>::clear(v_tile(buf), VS, p.Dv, t);
  }
  stash(0);
  __syncthreads();
  int cur = 0;
  for (int it = 0; it < ntiles; it++) {
    bool const more = it + 1 < ntiles;
    if (more) fetch((it + 1) * C::kT);
#pragma unroll
    for (int j = 0; j < J; j++) {
      int const kt0 = it * C::kT + (kw * J + j) * 32;
      bool const active = kt0 < p.Skv && (!p.causal || kt0 <= qw0 + 31);
      if (!active) continue;
      bf16 const *kr = k_tile(cur) + (kw * J + j) * 32 * KS;
      bf16 const *kk_ = kr + koff, *vk_ = v_tile(cur) + (kw * J + j) * 32 * VS + voff, *ktr = kr + toff;
      // S^T = K Q^T, dP^T = V dO^T: rows = keys, column = this lane's query
      f32x16 s, dp;
#pragma unroll
      for (int r = 0; r < 16; r++) {
        s[r] = 0.0f;
        dp[r] = 0.0f;
      }
#pragma unroll
      for (int kk = 0; kk < DP / 16; kk++) {
        bf16x8 const ka = frag_k(kk_, KS, 0, kk * 16);
        s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka, qf[kk], s, 0, 0, 0);
        bf16x8 const va = frag_k(vk_, VS, 0, kk * 16);
        dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, gf[kk], dp, 0, 0, 0);
      }
      float dsv[16];
#pragma unroll
      for (int r = 0; r < 16; r++) {
        float const e = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], p.scale_log2, -lse2));
        dsv[r] = e * __builtin_fmaf(dp[r], p.scale, -delta_s);
      }
      if (kt0 + 32 > p.Skv || (p.causal && kt0 + 31 > qw0)) {
#pragma unroll
        for (int r = 0; r < 16; r++) {
          int const kv = kt0 + 8 * (r >> 2) + 4 * h32 + (r & 3);
          dsv[r] = kv >= p.Skv || (p.causal && kv > qrow) ? 0.0f : dsv[r];
        }
      }
      // dQ^T += K^T dS^T: A = K^T (rows d) through transposing loads, B = dS^T
#pragma unroll
      for (int s2 = 0; s2 < 2; s2++) {
        bf16x8 const db = pack8(dsv + 8 * s2);
#pragma unroll
        for (int i = 0; i < DP / 32; i++) {
          bf16x8 const ka = frag_tr_acc(ktr, KS, 0, s2, i * 32);
          dq[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka, db, dq[i], 0, 0, 0);
        }
      }
    }
    if (C::kBuffers == 1) __syncthreads();
    if (more) stash(C::kBuffers == 1 ? 0 : cur ^ 1);
    __syncthreads();
    if (C::kBuffers == 2) cur ^= 1;
  }

  if constexpr (KW > 1) {
    float *const slots = reinterpret_cast<float *>(pool) + qw * (KW - 1) * DP * 32;
    if (kw > 0) gen_put<DP / 32>(slots + (kw - 1) * DP * 32, dq, lane);
    __syncthreads();
    if (kw > 0) return;
#pragma unroll
    for (int w = 0; w < KW - 1; w++) gen_add<DP / 32>(slots + w * DP * 32, 1.0f, dq, lane);
  }
  if (qrow < p.Sq) {
    bf16 *dqp = p.dq + (int64_t)b * p.q_bs + (int64_t)qrow * p.q_ss + (int64_t)head * p.Dq;
#pragma unroll
    for (int i = 0; i < DP / 32; i++) {
#pragma unroll
      for (int g = 0; g < 4; g++) {
        int const d = i * 32 + 8 * g + 4 * h32;
        if (d < p.Dq) {
          u32x2 w = {pack_bf16x2(dq[i][4 * g], dq[i][4 * g + 1]), pack_bf16x2(dq[i][4 * g + 2], dq[i][4 * g + 3])};
          *reinterpret_cast<u32x2 *>(dqp + d) = w;
        }
      }
    }
  }
}

// --------------------------------------------------------------------------
// backward (A): dK, dV.
// --------------------------------------------------------------------------
// Accumulators with rows = keys (8*(r/4) + 4*h + r%4 of this wave's 32), column = d, so a
// lane holds one column of 16 rows.  A wave turns its 32 x DP block around in LDS (the
// streamed tiles are done with) and writes whole 16-byte pieces of the first `rows` rows.
template <int DP>
__device__ __forceinline__ void gen_write_out(bf16 *stage, f32x16 const (&acc)[DP / 32], bf16 *out, int64_t row_stride,
                                              int D, int rows, int lane) {
  constexpr int OS = DP + 8;
  int const h32 = lane >> 5;
#pragma unroll
  for (int i = 0; i < DP / 32; i++) {
#pragma unroll
    for (int r = 0; r < 16; r++) {
      int const row = 8 * (r >> 2) + 4 * h32 + (r & 3);
      VecIO<bf16>::store1(stage + row * OS + i * 32 + (lane & 31), acc[i][r]);
    }
  }
  // LDS operations of one wave complete in order: the reads below see the writes above
#pragma unroll
  for (int k = 0; k < 32 * (DP / 8) / 64; k++) {
    int const c = lane + k * 64;
    int const row = c / (DP / 8), ch = c % (DP / 8);
    u32x4 const v = *reinterpret_cast<u32x4 const *>(stage + row * OS + ch * 8);
    if (row < rows && ch * 8 < D) *reinterpret_cast<u32x4 *>(out + (int64_t)row * row_stride + ch * 8) = v;
  }
}

// Head sizes up to 96: a wave computes scores and dP of its keys and accumulates both gradients.
// workgroup = 128 / KW keys.
template <int DP, int KW>
struct GenDkdv {
  static constexpr int kJ = KW == 1 ? 2 : 1;  // 32-query blocks of a wave and step
  static constexpr int kT = 32 * kJ * KW;
  static constexpr int kStride = GenStride<DP>::both;
  static constexpr int kTile = 2 * kT * kStride;  // elements, Q and dO
  static constexpr int kBuffers = 2 * kTile * 2 <= kGenLds ? 2 : 1;
  static constexpr int kOut = 4 / KW * 32 * (DP + 8) * 2;               // bytes, of the waves that write out
  static constexpr int kMerge = (KW - 1) * (4 / KW) * 2 * DP * 32 * 4;
  static constexpr int kBytes0 = kBuffers * kTile * 2 > kOut ? kBuffers * kTile * 2 : kOut;
  static constexpr int kBytes = kBytes0 > kMerge ? kBytes0 : kMerge;
};
template <int DP, int KW>
__global__ __launch_bounds__(256) void attn_gen_bwd_dkdv_kernel(AttnGenParams p) {
  using C = GenDkdv<DP, KW>;
  constexpr int S = C::kStride, KR = 128 / KW, J = C::kJ;
  __shared__ __attribute__((aligned(16))) uint8_t pool[C::kBytes];
  __shared__ __attribute__((aligned(16))) float Ls[C::kBuffers][C::kT], Ds[C::kBuffers][C::kT];
  int const t = threadIdx.x, lane = t & 63, h32 = lane >> 5;
  int const wave = __builtin_amdgcn_readfirstlane(t >> 6);
  int const kg = wave / KW, kw = wave % KW;
  int const hb = blockIdx.x % (p.H * p.B);
  int const head = hb % p.H, b = hb / p.H;
  int const kv0 = (blockIdx.x / (p.H * p.B)) * KR, kv0w = kv0 + kg * 32;
  int const kvrow = kv0w + (lane & 31);
  bf16 const *qp = p.q + (int64_t)b * p.q_bs + (int64_t)head * p.Dq;
  bf16 const *gp = p.d_o + (int64_t)b * p.o_bs + (int64_t)head * p.Dv;
  bf16 const *kp = p.k + (int64_t)b * p.k_bs + (int64_t)head * p.Dq;
  bf16 const *vp = p.v + (int64_t)b * p.v_bs + (int64_t)head * p.Dv;
  float const *lsep = p.lse + ((int64_t)b * p.H + head) * p.Sq;
  float const *delp = p.delta + ((int64_t)b * p.H + head) * p.Sq;
  auto q_tile = [&](int buf) { return reinterpret_cast<bf16 *>(pool) + buf * C::kTile; };
  auto g_tile = [&](int buf) { return q_tile(buf) + C::kT * S; };

  int const q_begin = p.causal ? (kv0 / C::kT) * C::kT : 0;
  int const ntiles = q_begin < p.Sq ? (p.Sq - q_begin + C::kT - 1) / C::kT : 0;
  GenTile<DP, C::kT> tq, tg;
  float rl = 0.0f, rd = 0.0f;
  auto fetch = [&](int qt0) {
    tq.load(qp, p.q_ss, qt0, p.Sq - 1, p.Dq, t);
    tg.load(gp, p.o_ss, qt0, p.Sq - 1, p.Dv, t);
    int const gr = min(qt0 + (t & (C::kT - 1)), p.Sq - 1);
    rl = lsep[gr] * kLog2e;
    rd = delp[gr] * p.scale;  // delta * scale, so dS is one fma and one multiply per element
  };
  auto stash = [&](int buf) {
    tq.store(q_tile(buf), S, p.Dq, t);
    tg.store(g_tile(buf), S, p.Dv, t);
    if (t < C::kT) {
      Ls[buf][t] = rl;
      Ds[buf][t] = rd;
    }
  };
  if (ntiles > 0) fetch(q_begin);
  bf16x8 kf[DP / 16], vf[DP / 16];
  gen_load_owned<DP>(kp + (int64_t)min(kvrow, p.Skv - 1) * p.k_ss, p.Dq, h32, kf);
  gen_load_owned<DP>(vp + (int64_t)min(kvrow, p.Skv - 1) * p.v_ss, p.Dv, h32, vf);
  f32x16 dk[DP / 32], dv[DP / 32];
#pragma unroll
  for (int i = 0; i < DP / 32; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) {
      dk[i][r] = 0.0f;
      dv[i][r] = 0.0f;
    }

  int const koff = lane_k_off(S, lane);
  int const toff = lane_tr_off(S, lane);
#pragma unroll
  for (int buf = 0; buf < C::kBuffers; buf++) {
    GenTile<DP, C::kT>::clear(q_tile(buf), S, p.Dq, t);
    GenTile<DP, C::kT>::clear(g_tile(buf), S, p.Dv, t);
  }
  if (ntiles > 0) stash(0);
  __syncthreads();
  int cur = 0;
  for (int it = 0; it < ntiles; it++) {
    bool const more = it + 1 < ntiles;
    if (more) fetch(q_begin + (it + 1) * C::kT);
#pragma unroll
    for (int j = 0; j < J; j++) {
      int const row0 = (kw * J + j) * 32, qt0 = q_begin + it * C::kT + row0;
      // keys that all lie after these queries (causal), or queries that do not exist, contribute nothing
      if (qt0 >= p.Sq || (p.causal && kv0w > qt0 + 31)) continue;
      bf16 const *const qt = q_tile(cur) + row0 * S, *const gt = g_tile(cur) + row0 * S;
      // S = Q K^T and dP = dO V^T: rows = queries of the tile, column = this lane's key
      f32x16 s, dp;
#pragma unroll
      for (int r = 0; r < 16; r++) {
        s[r] = 0.0f;
        dp[r] = 0.0f;
      }
#pragma unroll
      for (int kk = 0; kk < DP / 16; kk++) {
        s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag_k(qt + koff, S, 0, kk * 16), kf[kk], s, 0, 0, 0);
        dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag_k(gt + koff, S, 0, kk * 16), vf[kk], dp, 0, 0, 0);
      }
      float pv[16], dsv[16];
#pragma unroll
      for (int g = 0; g < 4; g++) {
        f32x4 const l = *reinterpret_cast<f32x4 const *>(&Ls[cur][row0 + 8 * g + 4 * h32]);
        f32x4 const d = *reinterpret_cast<f32x4 const *>(&Ds[cur][row0 + 8 * g + 4 * h32]);
#pragma unroll
        for (int e = 0; e < 4; e++) {
          int const r = 4 * g + e;
          pv[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], p.scale_log2, -l[e]));
          dsv[r] = pv[r] * __builtin_fmaf(dp[r], p.scale, -d[e]);  // dS = P (dP - delta) scale
        }
      }
      if (qt0 + 32 > p.Sq || kv0w + 32 > p.Skv || (p.causal && kv0w + 31 > qt0)) {
#pragma unroll
        for (int r = 0; r < 16; r++) {
          int const qg = qt0 + 8 * (r >> 2) + 4 * h32 + (r & 3);
          bool const masked = qg >= p.Sq || kvrow >= p.Skv || (p.causal && kvrow > qg);
          pv[r] = masked ? 0.0f : pv[r];
          dsv[r] = masked ? 0.0f : dsv[r];
        }
      }
      // dV += P^T dO ; dK += dS^T Q.  A = the accumulator re-used (row = key), B = dO / Q read
      // with the matching reduction order (k = query)
#pragma unroll
      for (int s2 = 0; s2 < 2; s2++) {
        bf16x8 const pa = pack8(pv + 8 * s2);
        bf16x8 const da = pack8(dsv + 8 * s2);
#pragma unroll
        for (int i = 0; i < DP / 32; i++) {
          dv[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(pa, frag_tr_acc(gt + toff, S, 0, s2, i * 32), dv[i], 0, 0, 0);
          dk[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(da, frag_tr_acc(qt + toff, S, 0, s2, i * 32), dk[i], 0, 0, 0);
        }
      }
    }
    if (C::kBuffers == 1) __syncthreads();
    if (more) stash(C::kBuffers == 1 ? 0 : cur ^ 1);
    __syncthreads();
    if (C::kBuffers == 2) cur ^= 1;
  }

  if constexpr (KW > 1) {
    float *const slots = reinterpret_cast<float *>(pool) + kg * (KW - 1) * 2 * DP * 32;
    if (kw > 0) {
      gen_put<DP / 32>(slots + (kw - 1) * 2 * DP * 32, dk, lane);
      gen_put<DP / 32>(slots + ((kw - 1) * 2 + 1) * DP * 32, dv, lane);
    }
    __syncthreads();
    if (kw == 0) {
#pragma unroll
      for (int w = 0; w < KW - 1; w++) {
        gen_add<DP / 32>(slots + w * 2 * DP * 32, 1.0f, dk, lane);
        gen_add<DP / 32>(slots + (w * 2 + 1) * DP * 32, 1.0f, dv, lane);
      }
    }
    __syncthreads();
    if (kw > 0) return;
  }
  bf16 *const stage = reinterpret_cast<bf16 *>(pool) + kg * 32 * (DP + 8);
  int64_t const row0 = (int64_t)kv0w;
  gen_write_out<DP>(stage, dk, p.dk + (int64_t)b * p.k_bs + row0 * p.k_ss + (int64_t)head * p.Dq, p.k_ss, p.Dq, p.Skv - kv0w, lane);
  gen_write_out<DP>(stage, dv, p.dv + (int64_t)b * p.v_bs + row0 * p.v_ss + (int64_t)head * p.Dv, p.v_ss, p.Dv, p.Skv - kv0w, lane);
}

// Larger head sizes: waves work in pairs on the same 32 keys, all that a workgroup owns.  One computes the scores
// and the probabilities and accumulates dV, the other dP, from which with the first one's probabilities (through
// LDS, 32 bits) dS, and dK.  Either holds one operand's fragments and one accumulator, so a head size of 256 fits
// the registers and is one launch with nothing computed twice.
template <int DP>
struct GenPairs {
  static constexpr int kT = 64;  // queries of a step, 32 a pair
  static constexpr int kStride = GenStride<DP>::both;
  static constexpr int kTile = 2 * kT * kStride;  // elements, Q and dO
  static constexpr int kBuffers = 2 * kTile * 2 <= kGenLds ? 2 : 1;
  static constexpr int kMerge = 2 * DP * 32 * 4;  // bytes; more than the waves that write out need
  static constexpr int kBytes = kBuffers * kTile * 2 > kMerge ? kBuffers * kTile * 2 : kMerge;
};
template <int DP>
__global__ __launch_bounds__(256) void attn_gen_bwd_dkdv_pairs_kernel(AttnGenParams p) {
  using C = GenPairs<DP>;
  constexpr int S = C::kStride;
  __shared__ __attribute__((aligned(16))) uint8_t pool[C::kBytes];
  __shared__ __attribute__((aligned(16))) float probs[2][32 * 32];  // of a pair
  __shared__ __attribute__((aligned(16))) float Ls[C::kBuffers][C::kT], Ds[C::kBuffers][C::kT];
  int const t = threadIdx.x, lane = t & 63, h32 = lane >> 5;
  int const wave = __builtin_amdgcn_readfirstlane(t >> 6);
  int const pair = wave >> 1;
  bool const is_k = (wave & 1) != 0;  // the one that makes dK
  int const hb = blockIdx.x % (p.H * p.B);
  int const head = hb % p.H, b = hb / p.H;
  int const kv0 = (blockIdx.x / (p.H * p.B)) * 32;
  int const kvrow = kv0 + (lane & 31);
  bf16 const *qp = p.q + (int64_t)b * p.q_bs + (int64_t)head * p.Dq;
  bf16 const *gp = p.d_o + (int64_t)b * p.o_bs + (int64_t)head * p.Dv;
  bf16 const *kp = p.k + (int64_t)b * p.k_bs + (int64_t)head * p.Dq;
  bf16 const *vp = p.v + (int64_t)b * p.v_bs + (int64_t)head * p.Dv;
  float const *lsep = p.lse + ((int64_t)b * p.H + head) * p.Sq;
  float const *delp = p.delta + ((int64_t)b * p.H + head) * p.Sq;
  auto q_tile = [&](int buf) { return reinterpret_cast<bf16 *>(pool) + buf * C::kTile; };
  auto g_tile = [&](int buf) { return q_tile(buf) + C::kT * S; };

  int const q_begin = p.causal ? (kv0 / C::kT) * C::kT : 0;
  int const ntiles = q_begin < p.Sq ? (p.Sq - q_begin + C::kT - 1) / C::kT : 0;
  GenTile<DP, C::kT> tq, tg;
  float rl = 0.0f, rd = 0.0f;
  auto fetch = [&](int qt0) {
    tq.load(qp, p.q_ss, qt0, p.Sq - 1, p.Dq, t);
    tg.load(gp, p.o_ss, qt0, p.Sq - 1, p.Dv, t);
    int const gr = min(qt0 + (t & (C::kT - 1)), p.Sq - 1);
    rl = lsep[gr] * kLog2e;
    rd = delp[gr] * p.scale;  // delta * scale, so dS is one fma and one multiply per element
  };
  auto stash = [&](int buf) {
    tq.store(q_tile(buf), S, p.Dq, t);
    tg.store(g_tile(buf), S, p.Dv, t);
    if (t < C::kT) {
      Ls[buf][t] = rl;
      Ds[buf][t] = rd;
    }
  };
  if (ntiles > 0) fetch(q_begin);
  bf16x8 own[DP / 16];  // this lane's row of K, or of V
  {
    int64_t const r = min(kvrow, p.Skv - 1);
    gen_load_owned<DP>(is_k ? vp + r * p.v_ss : kp + r * p.k_ss, is_k ? p.Dv : p.Dq, h32, own);
  }
  f32x16 acc[DP / 32];
#pragma unroll
  for (int i = 0; i < DP / 32; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) acc[i][r] = 0.0f;

  int const koff = lane_k_off(S, lane);
  int const toff = lane_tr_off(S, lane);
#pragma unroll
  for (int buf = 0; buf < C::kBuffers; buf++) {
    GenTile<DP, C::kT>::clear(q_tile(buf), S, p.Dq, t);
    GenTile<DP, C::kT>::clear(g_tile(buf), S, p.Dv, t);
  }
  if (ntiles > 0) stash(0);
  __syncthreads();
  int cur = 0;
  for (int it = 0; it < ntiles; it++) {
    bool const more = it + 1 < ntiles;
    if (more) fetch(q_begin + (it + 1) * C::kT);
    // S = Q K^T, or dP = dO V^T: rows = queries of the tile, column = this lane's key
    f32x16 z;
    float w[16];
    int const row0 = pair * 32, qt0 = q_begin + it * C::kT + row0;
    // keys that all lie after these queries (causal), or queries that do not exist, contribute nothing
    bool const active = qt0 < p.Sq && (!p.causal || kv0 <= qt0 + 31);
    if (active) {
      bf16 const *const x = (is_k ? g_tile(cur) : q_tile(cur)) + row0 * S + koff;
#pragma unroll
      for (int r = 0; r < 16; r++) z[r] = 0.0f;
#pragma unroll
      for (int kk = 0; kk < DP / 16; kk++) {
        z = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag_k(x, S, 0, kk * 16), own[kk], z, 0, 0, 0);
      }
      if (!is_k) {
        bool const edge = qt0 + 32 > p.Sq || kv0 + 32 > p.Skv || (p.causal && kv0 + 31 > qt0);
#pragma unroll
        for (int g = 0; g < 4; g++) {
          f32x4 const l = *reinterpret_cast<f32x4 const *>(&Ls[cur][row0 + 8 * g + 4 * h32]);
#pragma unroll
          for (int e = 0; e < 4; e++) {
            w[4 * g + e] = __builtin_amdgcn_exp2f(__builtin_fmaf(z[4 * g + e], p.scale_log2, -l[e]));
          }
        }
        if (edge) {
#pragma unroll
          for (int r = 0; r < 16; r++) {
            int const qg = qt0 + 8 * (r >> 2) + 4 * h32 + (r & 3);
            w[r] = qg >= p.Sq || kvrow >= p.Skv || (p.causal && kvrow > qg) ? -0.0f : w[r];
          }
        }
#pragma unroll
        for (int g = 0; g < 4; g++) {
          *reinterpret_cast<f32x4 *>(&probs[pair][(g * 64 + lane) * 4]) =
              f32x4{w[4 * g], w[4 * g + 1], w[4 * g + 2], w[4 * g + 3]};
        }
      }
    }
    __syncthreads();
    if (active) {
      if (is_k) {
#pragma unroll
        for (int g = 0; g < 4; g++) {
          f32x4 const pv = *reinterpret_cast<f32x4 const *>(&probs[pair][(g * 64 + lane) * 4]);
          f32x4 const d = *reinterpret_cast<f32x4 const *>(&Ds[cur][row0 + 8 * g + 4 * h32]);
          // dS = P (dP - delta) scale; -0 is what the other wave has put where P is masked
#pragma unroll
          for (int e = 0; e < 4; e++) {
            w[4 * g + e] =
                __float_as_uint(pv[e]) == 0x80000000u ? 0.0f : pv[e] * __builtin_fmaf(z[4 * g + e], p.scale, -d[e]);
          }
        }
      }
      // dV += P^T dO, or dK += dS^T Q: A = the accumulator re-used (row = key), B = dO / Q read with the
      // matching reduction order (k = query)
      bf16 const *const y = (is_k ? q_tile(cur) : g_tile(cur)) + row0 * S + toff;
#pragma unroll
      for (int s2 = 0; s2 < 2; s2++) {
        bf16x8 const a = pack8(w + 8 * s2);
#pragma unroll
        for (int i = 0; i < DP / 32; i++) {
          acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, frag_tr_acc(y, S, 0, s2, i * 32), acc[i], 0, 0, 0);
        }
      }
    }
    if (C::kBuffers == 1) __syncthreads();
    if (more) stash(C::kBuffers == 1 ? 0 : cur ^ 1);
    __syncthreads();
    if (C::kBuffers == 2) cur ^= 1;
  }

  float *const slot = reinterpret_cast<float *>(pool) + (wave & 1) * DP * 32;
  if (pair > 0) gen_put<DP / 32>(slot, acc, lane);
  __syncthreads();
  if (pair == 0) gen_add<DP / 32>(slot, 1.0f, acc, lane);
  __syncthreads();
  if (pair > 0) return;
  bf16 *const stage = reinterpret_cast<bf16 *>(pool) + (wave & 1) * 32 * (DP + 8);
  int64_t const row0 = (int64_t)kv0;
  if (is_k) gen_write_out<DP>(stage, acc, p.dk + (int64_t)b * p.k_bs + row0 * p.k_ss + (int64_t)head * p.Dq, p.k_ss, p.Dq, p.Skv - kv0, lane);
  else gen_write_out<DP>(stage, acc, p.dv + (int64_t)b * p.v_bs + row0 * p.v_ss + (int64_t)head * p.Dv, p.v_ss, p.Dv, p.Skv - kv0, lane);
}

static int check_desc_gen(char const *who, ffk_attention_desc_t const *d) {
  int64_t const dq = d->head_dim, dv = d->v_head_dim > 0 ? d->v_head_dim : d->head_dim;
  FFK_REQUIRE(dq > 0 && dq <= 256 && dq % 8 == 0 && dv <= 256 && dv % 8 == 0,
              "%s: bf16 head_dim %lld / v_head_dim %lld not supported (multiples of 8 up to 256)", who,
              (long long)dq, (long long)dv);
  FFK_REQUIRE(d->q_seq_stride >= d->heads * dq && d->k_seq_stride >= d->heads * dq &&
                  d->v_seq_stride >= d->heads * dv && d->o_seq_stride >= d->heads * dv,
              "%s: sequence stride smaller than heads * head_dim", who);
  return FFK_OK;
}

static AttnGenParams make_gen_params(ffk_attention_desc_t const *d) {
  AttnGenParams p = {};
  p.B = (int)d->batch; p.H = (int)d->heads; p.Sq = (int)d->seq_q; p.Skv = (int)d->seq_kv;
  p.Dq = (int)d->head_dim;
  p.Dv = (int)(d->v_head_dim > 0 ? d->v_head_dim : d->head_dim);
  p.q_bs = d->q_batch_stride; p.q_ss = d->q_seq_stride;
  p.k_bs = d->k_batch_stride; p.k_ss = d->k_seq_stride;
  p.v_bs = d->v_batch_stride; p.v_ss = d->v_seq_stride;
  p.o_bs = d->o_batch_stride; p.o_ss = d->o_seq_stride;
  p.scale = d->scale;
  p.scale_log2 = d->scale * kLog2e;
  p.causal = d->causal;
  return p;
}

#define FFK_ATTN_GEN_DISPATCH(D_, CALL)                                        \
  do {                                                                         \
    if ((D_) <= 32) { CALL(32); }                                              \
    else if ((D_) <= 64) { CALL(64); }                                         \
    else if ((D_) <= 96) { CALL(96); }                                         \
    else if ((D_) <= 128) { CALL(128); }                                       \
    else { CALL(256); }                                                        \
  } while (0)

// How many waves share a group's rows, up to `most`: the fewest that give the chip `enough` workgroups.  (times in
// us by KW = 1, 2, 4; 4 heads: [B, S, D] forward / dQ / dK and dV)
//   [2, 1198, 64]  80 WGs   27 19 20 / 34 23 22 / 57 36 30     [3, 390, 80]   96 WGs   15 12 20 / 17 15 16 / 24 18 28
//   [8, 600, 32]  160 WGs   14  9  8 / 15 11 10 / 18 13 10     [4, 798, 256] 112 WGs   55 39  - / 68 45  -
//   [16, 403, 80] 256 WGs   17 25 41 / 19 21 31 / 26 36 58     [48, 600, 32] 960 WGs   30 33 38 / 33 39 47 / 48 51 61
// At a head size of 32 two workgroups a CU are not too many.  ([64, 512, 256] 256 WGs: 45 64 - / 58 76 -, [20, 2297, 256]
// 360: 305 331 - / 376 360 -.)
static int gen_split(AttnGenParams const &p, int rows, int streamed, int most, int enough) {
  int kw = 1;
  while (kw < most && (int64_t)p.H * p.B * ceil_div(rows, 128 / kw) < enough && streamed > 32 * kw) kw *= 2;
  return kw;
}
template <int DP>
constexpr int kGenEnough = DP == 32 ? 2 * kNumCU : kNumCU;

template <int DP>
static void launch_gen_forward(hipStream_t st, AttnGenParams const &p) {
  int const kw = gen_split(p, p.Sq, p.Skv, DP == 32 ? 4 : 2, kGenEnough<DP>);
  unsigned const grid = (unsigned)(ceil_div(p.Sq, 128 / kw) * p.H * p.B);
  if constexpr (DP == 32) {
    if (kw == 4) return (void)(attn_gen_fwd_kernel<DP, 4><<<grid, 256, 0, st>>>(p));
  }
  if (kw == 2) attn_gen_fwd_kernel<DP, 2><<<grid, 256, 0, st>>>(p);
  else attn_gen_fwd_kernel<DP, 1><<<grid, 256, 0, st>>>(p);
}

template <int DP>
static void launch_gen_dq(hipStream_t st, AttnGenParams const &p) {
  int const kw = gen_split(p, p.Sq, p.Skv, DP == 32 ? 4 : 2, kGenEnough<DP>);
  unsigned const grid = (unsigned)(ceil_div(p.Sq, 128 / kw) * p.H * p.B);
  if constexpr (DP == 32) {
    if (kw == 4) return (void)(attn_gen_bwd_dq_kernel<DP, 4><<<grid, 256, 0, st>>>(p));
  }
  if (kw == 2) attn_gen_bwd_dq_kernel<DP, 2><<<grid, 256, 0, st>>>(p);
  else attn_gen_bwd_dq_kernel<DP, 1><<<grid, 256, 0, st>>>(p);
}

template <int DP>
static void launch_gen_dkdv(hipStream_t st, AttnGenParams const &p) {
  if constexpr (DP <= 96) {
    int const kw = gen_split(p, p.Skv, p.Sq, DP <= 64 ? 4 : 2, kGenEnough<DP>);
    unsigned const grid = (unsigned)(ceil_div(p.Skv, 128 / kw) * p.H * p.B);
    if constexpr (DP <= 64) {
      if (kw == 4) return (void)(attn_gen_bwd_dkdv_kernel<DP, 4><<<grid, 256, 0, st>>>(p));
    }
    if (kw == 2) attn_gen_bwd_dkdv_kernel<DP, 2><<<grid, 256, 0, st>>>(p);
    else attn_gen_bwd_dkdv_kernel<DP, 1><<<grid, 256, 0, st>>>(p);
  } else {
    attn_gen_bwd_dkdv_pairs_kernel<DP><<<(unsigned)(ceil_div(p.Skv, 32) * p.H * p.B), 256, 0, st>>>(p);
  }
}

// shapes, strides and alignment other than the head sizes are checked by the caller (attention.hip)
int attention_bf16_general_forward(hipStream_t st, ffk_attention_desc_t const *d, void const *q, void const *k,
                                   void const *v, void *o, float *lse) {
  int rc = check_desc_gen("attention_forward", d);
  if (rc != FFK_OK) return rc;
  AttnGenParams p = make_gen_params(d);
  p.q = static_cast<bf16 const *>(q);
  p.k = static_cast<bf16 const *>(k);
  p.v = static_cast<bf16 const *>(v);
  p.out = static_cast<bf16 *>(o);
  p.lse = lse;
  int const dmax = p.Dq > p.Dv ? p.Dq : p.Dv;
#define CALL(DP_) launch_gen_forward<DP_>(st, p)
  FFK_ATTN_GEN_DISPATCH(dmax, CALL);
#undef CALL
  FFK_CHECK_LAUNCH();
  return FFK_OK;
}

int attention_bf16_general_backward(hipStream_t st, ffk_attention_desc_t const *d, void const *q, void const *k,
                                    void const *v, void const *o, void const *d_o, float const *lse,
                                    float *delta, void *dq, void *dk, void *dv, int what) {
  int rc = check_desc_gen("attention_backward", d);
  if (rc != FFK_OK) return rc;
  AttnGenParams p = make_gen_params(d);
  p.q = static_cast<bf16 const *>(q);
  p.k = static_cast<bf16 const *>(k);
  p.v = static_cast<bf16 const *>(v);
  p.o = static_cast<bf16 const *>(o);
  p.d_o = static_cast<bf16 const *>(d_o);
  p.lse = const_cast<float *>(lse);
  p.delta = delta;
  p.dq = static_cast<bf16 *>(dq);
  p.dk = static_cast<bf16 *>(dk);
  p.dv = static_cast<bf16 *>(dv);
  int const dmax = p.Dq > p.Dv ? p.Dq : p.Dv;
  // dQ first: it leaves delta in memory for the dK/dV kernel
#define CALL(DP_)                                                              \
  do {                                                                         \
    if ((what & 1) != 0) launch_gen_dq<DP_>(st, p);                            \
    if ((what & 2) != 0) launch_gen_dkdv<DP_>(st, p);                          \
  } while (0)
  FFK_ATTN_GEN_DISPATCH(dmax, CALL);
#undef CALL
  FFK_CHECK_LAUNCH();
  return FFK_OK;
}

}  // namespace ffk
