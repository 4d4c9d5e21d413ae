// Stable least-significant-digit radix sort of (row id, lookup number) pairs
// on the device, for the sorted embedding backward: rows that are looked up
// several times end up next to each other, in ascending lookup order.
//
// One pass sorts by 8 bits of the key and is three launches:
//   histogram  a workgroup counts the digits of its tile of 2048 keys into
//              table[digit][tile] and adds them to the digit totals of the pass;
//   scan       workgroup d turns row d of the table into exclusive prefix sums
//              on top of the totals of the digits below d: entry (d, t) becomes
//              the first output position of tile t's keys with digit d;
//   scatter    the workgroup re-reads its tile; each of its four waves owns a
//              quarter of it and walks that quarter 64 keys at a time in order,
//              ranking the keys of a step among their peers with the same digit
//              by ballots, so equal digits keep their input order (stable) and
//              the result does not depend on timing (no atomics decide a place).
// Up to 1 048 576 lookups a pass is one to three launches: the scan moves into the scatter
// kernel (every workgroup adds up the counts of the tiles before its own and the
// totals of the digits below, straight from a table of at most 256 KB), and the
// scatter counts the NEXT pass's digits of the keys it places, per destination
// tile, with integer atomics (a count does not depend on the order of the
// additions; the counts are gathered in LDS first, since under a skewed id
// distribution thousands of a workgroup's keys share one counter), or beyond
// 131 072 lookups a histogram launch does.  Digits are as
// narrow as the number of passes allows, and up to ten bits wide where that saves a
// pass (radix_sort_plan).  Up to 4096 lookups the whole sort is one workgroup and one launch.
// The first pass reads the caller's index tensor directly (int32 or int64,
// ids outside the table become the key `invalid_key`, which sorts behind every
// row) and numbers the lookups itself, so no pass exists only to build keys.
#pragma once
#include "ffk_common.h"

namespace ffk {

constexpr int kSortThreads = 256;
constexpr int kSortItems = 8;                              // keys per thread
constexpr int kSortTile = kSortThreads * kSortItems;       // keys per workgroup
constexpr int kSortRadix = 256;
constexpr int kSortWaveKeys = kSortTile / 4;               // keys per wave

template <typename IT, bool FIRST>
__device__ __forceinline__ uint32_t sort_key_at(IT const *idx, uint32_t const *keys_in, int64_t i,
                                                int64_t num_entries) {
  if constexpr (FIRST) {
    int64_t const r = (int64_t)idx[i];
    return (uint64_t)r < (uint64_t)num_entries ? (uint32_t)r : (uint32_t)num_entries;
  } else {
    return keys_in[i];
  }
}

template <typename IT, bool FIRST>
__global__ __launch_bounds__(kSortThreads) void radix_hist_kernel(IT const *__restrict__ idx,
                                                                  uint32_t const *__restrict__ keys_in,
                                                                  uint32_t *__restrict__ table,
                                                                  uint32_t *__restrict__ totals, int64_t n,
                                                                  int ntiles, int shift, int64_t num_entries) {
  __shared__ uint32_t cnt[kSortRadix];
  cnt[threadIdx.x] = 0;
  __syncthreads();
  int64_t const base = (int64_t)blockIdx.x * kSortTile;
#pragma unroll
  for (int k = 0; k < kSortItems; k++) {
    int64_t const i = base + k * kSortThreads + threadIdx.x;
    if (i < n) {
      uint32_t const key = sort_key_at<IT, FIRST>(idx, keys_in, i, num_entries);
      atomicAdd(&cnt[(key >> shift) & (kSortRadix - 1)], 1u);  // LDS; a count does not depend on order
    }
  }
  __syncthreads();
  uint32_t const c = cnt[threadIdx.x];
  table[(int64_t)threadIdx.x * ntiles + blockIdx.x] = c;
  if (c != 0) atomicAdd(&totals[threadIdx.x], c);  // integer sums: the order of the additions does not matter
}

__global__ __launch_bounds__(256) void radix_zero_kernel(uint32_t *p, int count) {
  int const i = blockIdx.x * 256 + threadIdx.x;
  if (i < count) p[i] = 0;
}

// Workgroup d: row d of the table (ntiles counts) becomes exclusive prefix sums
// that start at the number of keys whose digit is below d.
__global__ __launch_bounds__(kSortThreads) void radix_scan_kernel(uint32_t *table, uint32_t const *__restrict__ totals,
                                                                  int ntiles) {
  __shared__ uint32_t wsum[4];
  int const t = threadIdx.x, lane = t & 63, wave = t >> 6, d = blockIdx.x;
  auto block_sum = [&](uint32_t v) {  // every thread gets the total
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    __syncthreads();  // wsum may still be read from the previous use
    if (lane == 0) wsum[wave] = v;
    __syncthreads();
    return wsum[0] + wsum[1] + wsum[2] + wsum[3];
  };
  uint32_t carry = block_sum(t < d ? totals[t] : 0u);
  uint32_t *row = table + (int64_t)d * ntiles;
  for (int c0 = 0; c0 < ntiles; c0 += kSortThreads) {
    int const i = c0 + t;
    uint32_t const x = i < ntiles ? row[i] : 0u;
    uint32_t incl = x;  // inclusive scan inside the wave
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      uint32_t const up = __shfl_up(incl, off, 64);
      if (lane >= off) incl += up;
    }
    __syncthreads();
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    uint32_t before = 0;
#pragma unroll
    for (int w = 0; w < 4; w++) before += w < wave ? wsum[w] : 0u;
    if (i < ntiles) row[i] = carry + before + incl - x;
    carry += wsum[0] + wsum[1] + wsum[2] + wsum[3];
  }
}

template <typename IT, bool FIRST>
__global__ __launch_bounds__(kSortThreads) void radix_scatter_kernel(
    IT const *__restrict__ idx, uint32_t const *__restrict__ keys_in, uint32_t const *__restrict__ vals_in,
    uint32_t *__restrict__ keys_out, uint32_t *__restrict__ vals_out, uint32_t const *__restrict__ table, int64_t n,
    int ntiles, int shift, int64_t num_entries) {
  __shared__ uint32_t wave_off[4][kSortRadix];  // per wave: digit counts, then the next free output position
  int const t = threadIdx.x, lane = t & 63, wave = t >> 6;
  for (int d = lane; d < kSortRadix; d += 64) wave_off[wave][d] = 0;
  // the zeroing above and the counting below touch this wave's row only, in program order
  int64_t const first = (int64_t)blockIdx.x * kSortTile + (int64_t)wave * kSortWaveKeys;
  constexpr int STEPS = kSortWaveKeys / 64;
  uint32_t key[STEPS], val[STEPS];
#pragma unroll
  for (int c = 0; c < STEPS; c++) {
    int64_t const i = first + c * 64 + lane;
    key[c] = 0;
    val[c] = 0;
    if (i < n) {
      key[c] = sort_key_at<IT, FIRST>(idx, keys_in, i, num_entries);
      val[c] = FIRST ? (uint32_t)i : vals_in[i];
      atomicAdd(&wave_off[wave][(key[c] >> shift) & (kSortRadix - 1)], 1u);
    }
  }
  __syncthreads();
  {
    // thread d: where each wave's keys with digit d start
    uint32_t run = table[(int64_t)t * ntiles + blockIdx.x];
#pragma unroll
    for (int w = 0; w < 4; w++) {
      uint32_t const c = wave_off[w][t];
      wave_off[w][t] = run;
      run += c;
    }
  }
  __syncthreads();
  uint64_t const below = ((uint64_t)1 << lane) - 1;
#pragma unroll
  for (int c = 0; c < STEPS; c++) {
    bool const valid = first + c * 64 + lane < n;
    uint32_t const digit = (key[c] >> shift) & (kSortRadix - 1);
    uint64_t peers = __ballot(valid);  // lanes of this step with this lane's digit
#pragma unroll
    for (int bit = 0; bit < 8; bit++) {
      uint64_t const m = __ballot((digit >> bit) & 1u);
      peers &= ((digit >> bit) & 1u) ? m : ~m;
    }
    if (valid) {
      uint32_t const start = wave_off[wave][digit];
      uint32_t const rank = (uint32_t)__popcll(peers & below);
      keys_out[start + rank] = key[c];
      vals_out[start + rank] = val[c];
      // LDS operations of a wave complete in program order: every peer has read `start`
      // before the first of them moves it on for the next step
      if (rank == 0) wave_off[wave][digit] = start + (uint32_t)__popcll(peers);
    }
  }
}

// ---------------------------------------------------------------------------
// One launch per pass, up to kSortFusedTiles tiles of 1024 threads with ITEMS
// keys each.  Tables are [tile][digit], one per pass (pass p's is filled by the
// histogram kernel for p = 0 and by pass p-1's scatter otherwise; each kernel
// clears the table that the kernel after it adds into, so no launch exists only
// to clear).  Bound by the latency of one workgroup's chain (keys, ranks, table,
// places), not by bandwidth, hence sixteen waves with at most four steps each,
// the ranking under the table's loads, and digits no wider than the passes need.
// Sort of 65 536 token ids below 50 257: 23 -> 18 us (tiles of 2048 keys and four
// waves before); 524 288 ids below a million: 63 -> 50 us (three launches a pass
// before), 40 in two passes of ten bits with a scan launch each; 1000 ids: three launches and 20 us less for the whole gradient.
// ---------------------------------------------------------------------------
constexpr int kSortFusedThreads = 1024;
constexpr int kSortFusedWaves = kSortFusedThreads / 64;
constexpr int kSortAheadTiles = 128;  // up to these a scatter counts the next pass's digits
constexpr int kSortFusedTiles = 256;
constexpr int kSortFusedItems = 4;  // the most keys per thread
constexpr int kSortWideRadix = 1024;
constexpr int kSortWideTiles = 16;

// A step's lanes with this lane's digit (all of them take part; `valid` lanes only are counted).
__device__ __forceinline__ uint64_t sort_peers(bool valid, uint32_t digit, int bits) {
  uint64_t peers = __ballot(valid);
  for (int bit = 0; bit < bits; bit++) {
    uint64_t const m = __ballot((digit >> bit) & 1u);
    peers &= ((digit >> bit) & 1u) ? m : ~m;
  }
  return peers;
}

// Place of each of a wave's keys among the wave's keys with the same digit, in
// input order; leaves the wave's digit counts in `count` (cleared by the caller).
template <int ITEMS>
__device__ __forceinline__ void sort_rank_wave(uint32_t const (&digit)[ITEMS], bool const (&valid)[ITEMS], int bits,
                                               int lane, uint32_t *count, uint32_t (&rank)[ITEMS]) {
  uint64_t const below = ((uint64_t)1 << lane) - 1;
#pragma unroll
  for (int c = 0; c < ITEMS; c++) {
    uint64_t const peers = sort_peers(valid[c], digit[c], bits);
    rank[c] = 0;
    if (valid[c]) {
      uint32_t const seen = count[digit[c]];
      uint32_t const r = (uint32_t)__popcll(peers & below);
      rank[c] = seen + r;
      // LDS operations of a wave complete in program order: every peer has read `seen`
      // before the first of them moves it on for the next step
      if (r == 0) count[digit[c]] = seen + (uint32_t)__popcll(peers);
    }
    __builtin_amdgcn_wave_barrier();  // the compiler keeps the next step's reads behind this
  }
}

// Exclusive prefix sum of v over the threads below `bins` (at most BINS; the others pass 0).
// Every thread calls it; it synchronises the workgroup once, on the way.
template <int BINS>
__device__ __forceinline__ uint32_t sort_scan_bins(uint32_t v, int t, int lane, uint32_t *wsum) {
  uint32_t incl = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    uint32_t const up = __shfl_up(incl, off, 64);
    if (lane >= off) incl += up;
  }
  if (lane == 63 && t < BINS) wsum[t >> 6] = incl;
  __syncthreads();
  uint32_t excl = incl - v;
#pragma unroll
  for (int w = 0; w < BINS / 64; w++) excl += w < (t >> 6) && t < BINS ? wsum[w] : 0u;
  return excl;
}

template <typename IT, bool FIRST, int BINS>
__global__ __launch_bounds__(kSortFusedThreads) void radix_hist_fused_kernel(IT const *__restrict__ idx,
                                                                            uint32_t const *__restrict__ keys_in,
                                                                            uint32_t *__restrict__ table0,
                                                                            uint32_t *__restrict__ table1, int64_t n,
                                                                            int items, int shift, int bits,
                                                                            int64_t num_entries) {
  __shared__ uint32_t cnt[BINS];
  int const t = threadIdx.x, bins = 1 << bits;
  if (t < BINS) cnt[t] = 0;
  __syncthreads();
  int64_t const base = (int64_t)blockIdx.x * kSortFusedThreads * items;
#pragma unroll
  for (int k = 0; k < kSortFusedItems; k++) {
    int64_t const i = base + k * kSortFusedThreads + t;
    if (k < items && i < n) {
      uint32_t const key = sort_key_at<IT, FIRST>(idx, keys_in, i, num_entries);
      atomicAdd(&cnt[(key >> shift) & (bins - 1)], 1u);  // LDS; a count does not depend on order
    }
  }
  __syncthreads();
  if (t < bins) {
    table0[(int64_t)blockIdx.x * bins + t] = cnt[t];
    if (table1 != nullptr) table1[(int64_t)blockIdx.x * bins + t] = 0;
  }
}

// table[tile][digit], counts, become the number of the digit's keys in the tiles before; totals[digit].
// A workgroup takes 64 digits, sixteen threads to each.
__global__ __launch_bounds__(kSortFusedThreads) void radix_scan_fused_kernel(uint32_t *table, uint32_t *__restrict__ totals,
                                                                            int ntiles, int bits) {
  constexpr int kParts = kSortFusedThreads / 64, kEach = kSortFusedTiles / kParts;
  __shared__ uint32_t part_sum[kParts][64];
  int const lane = threadIdx.x & 63, part = threadIdx.x >> 6, d = blockIdx.x * 64 + lane;
  uint32_t v[kEach], sum = 0;
#pragma unroll
  for (int k = 0; k < kEach; k++) {
    int const tile = part * kEach + k;
    v[k] = tile < ntiles ? table[((int64_t)tile << bits) + d] : 0u;
  }
#pragma unroll
  for (int k = 0; k < kEach; k++) sum += v[k];
  part_sum[part][lane] = sum;
  __syncthreads();
  uint32_t run = 0;
#pragma unroll
  for (int q = 0; q < kParts; q++) run += q < part ? part_sum[q][lane] : 0u;
#pragma unroll
  for (int k = 0; k < kEach; k++) {
    int const tile = part * kEach + k;
    if (tile < ntiles) table[((int64_t)tile << bits) + d] = run;
    run += v[k];
  }
  if (part == kParts - 1) totals[d] = run;
}

// table: this pass's counts; next: the next pass's table (nullptr on the last pass), added
// into here; after: the table of the pass after that (nullptr if none), cleared here.
// SCANNED: radix_scan_fused_kernel has been over the table, its totals behind it.
// Dynamic LDS: the workgroup's share of the next table, 16-bit counters in pairs (a workgroup
// counts its own keys there, at most 4096; only up to kSortAheadTiles tiles).
template <typename IT, bool FIRST, int ITEMS, int BINS, bool SCANNED>
__global__ __launch_bounds__(kSortFusedThreads) void radix_scatter_fused_kernel(
    IT const *__restrict__ idx, uint32_t const *__restrict__ keys_in, uint32_t const *__restrict__ vals_in,
    uint32_t *__restrict__ keys_out, uint32_t *__restrict__ vals_out, uint32_t const *__restrict__ table,
    uint32_t *__restrict__ next, uint32_t *__restrict__ after, int64_t n, int ntiles, int shift, int bits,
    int64_t num_entries) {
  constexpr int TILE = kSortFusedThreads * ITEMS;
  // pairs leave through LDS in order, where that makes runs of them
  constexpr bool kOrdered = ITEMS > 1 && BINS == kSortRadix;
  extern __shared__ uint32_t next_cnt[];
  __shared__ uint32_t wave_off[kSortFusedWaves][BINS];
  __shared__ uint32_t part_all[kSortFusedThreads], part_before[kSortFusedThreads];
  __shared__ uint32_t wsum[BINS / 64], delta[kOrdered ? BINS : 1];
  __shared__ uint32_t ks[kOrdered ? TILE : 1], vs[kOrdered ? TILE : 1];
  int const t = threadIdx.x, lane = t & 63, wave = t >> 6;
  int const bins = 1 << bits, mask = bins - 1;
  int const next_words = next != nullptr ? (ntiles * bins + 1) / 2 : 0;
  for (int d = lane; d < bins; d += 64) wave_off[wave][d] = 0;
  for (int i = t; i < next_words; i += kSortFusedThreads) next_cnt[i] = 0;
  int64_t const first = (int64_t)blockIdx.x * TILE + wave * (64 * ITEMS);
  uint32_t key[ITEMS], val[ITEMS], digit[ITEMS], rank[ITEMS];
  bool valid[ITEMS];
#pragma unroll
  for (int c = 0; c < ITEMS; c++) {
    int64_t const i = first + c * 64 + lane;
    valid[c] = i < n;
    key[c] = 0;
    val[c] = 0;
    if (valid[c]) {
      key[c] = sort_key_at<IT, FIRST>(idx, keys_in, i, num_entries);
      val[c] = FIRST ? (uint32_t)i : vals_in[i];
    }
  }
  // the keys with digit d in the tiles before this one, and in all tiles: 1024 / bins threads a digit
  if constexpr (SCANNED) {
    part_before[t] = t < bins ? table[((int64_t)blockIdx.x << bits) + t] : 0u;
    part_all[t] = t < bins ? table[((int64_t)ntiles << bits) + t] : 0u;
  } else {
    int const d = t & mask, part = t >> bits, parts = kSortFusedThreads >> bits, tile = blockIdx.x;
    uint32_t before_tiles = 0, all_tiles = 0;
    for (int t0 = part; t0 < ntiles; t0 += 16 * parts) {
      uint32_t v[16];
#pragma unroll
      for (int u = 0; u < 16; u++) v[u] = t0 + u * parts < ntiles ? table[(int64_t)(t0 + u * parts) * bins + d] : 0u;
#pragma unroll
      for (int u = 0; u < 16; u++) {
        all_tiles += v[u];
        before_tiles += t0 + u * parts < tile ? v[u] : 0u;
      }
    }
    part_all[t] = all_tiles;
    part_before[t] = before_tiles;
  }
  if (after != nullptr && t < bins) after[(int64_t)blockIdx.x * bins + t] = 0;
#pragma unroll
  for (int c = 0; c < ITEMS; c++) digit[c] = (key[c] >> shift) & mask;
  sort_rank_wave<ITEMS>(digit, valid, bits, lane, wave_off[wave], rank);
  __syncthreads();
  uint32_t all = 0, before = 0;
  if (t < bins) {
    for (int p = t; p < kSortFusedThreads; p += bins) {
      all += part_all[p];
      before += part_before[p];
    }
  }
  uint32_t const smaller = sort_scan_bins<BINS>(all, t, lane, wsum);
  if constexpr (!kOrdered) {
    if (t < bins) {
      uint32_t run = smaller + before;
#pragma unroll
      for (int w = 0; w < kSortFusedWaves; w++) {
        uint32_t const c = wave_off[w][t];
        wave_off[w][t] = run;
        run += c;
      }
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < ITEMS; c++) {
      if (valid[c]) {
        uint32_t const pos = wave_off[wave][digit[c]] + rank[c];
        keys_out[pos] = key[c];
        vals_out[pos] = val[c];
        // the next pass's count of this key, in the tile it has just been placed in
        if (next != nullptr) {
          uint32_t const nd = (pos / TILE) * bins + ((key[c] >> (shift + bits)) & mask);
          atomicAdd(&next_cnt[nd >> 1], 1u << (16 * (nd & 1u)));
        }
      }
    }
  } else {
    __syncthreads();
    // The pairs are put in order in LDS first and leave from there: a wave's stores then go to a few
    // runs of consecutive places instead of 64 lines (524 288 ids: 14 -> 12 us a pass; with one key a thread
    // the two more barriers cost more, 5.7 -> 7.3 us for 65 536).
    uint32_t mine = 0;
    if (t < bins) {
#pragma unroll
      for (int w = 0; w < kSortFusedWaves; w++) mine += wave_off[w][t];
    }
    uint32_t const local = sort_scan_bins<BINS>(mine, t, lane, wsum);
    if (t < bins) {
      delta[t] = smaller + before - local;  // from a pair's place in LDS to its place in the output
      uint32_t run = local;
#pragma unroll
      for (int w = 0; w < kSortFusedWaves; w++) {
        uint32_t const c = wave_off[w][t];
        wave_off[w][t] = run;
        run += c;
      }
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < ITEMS; c++) {
      if (valid[c]) {
        uint32_t const at = wave_off[wave][digit[c]] + rank[c];
        ks[at] = key[c];
        vs[at] = val[c];
      }
    }
    __syncthreads();
    int const here = (int)min((int64_t)TILE, n - (int64_t)blockIdx.x * TILE);
#pragma unroll
    for (int c = 0; c < ITEMS; c++) {
      int const at = c * kSortFusedThreads + t;
      if (at < here) {
        uint32_t const k = ks[at];
        uint32_t const pos = (uint32_t)at + delta[(k >> shift) & mask];
        keys_out[pos] = k;
        vals_out[pos] = vs[at];
      }
    }
  }
  if (next != nullptr) {
    __syncthreads();
    for (int i = t; i < next_words; i += kSortFusedThreads) {
      uint32_t const c = next_cnt[i];
      if ((c & 0xffffu) != 0) atomicAdd(&next[2 * (int64_t)i], c & 0xffffu);
      if ((c >> 16) != 0) atomicAdd(&next[2 * (int64_t)i + 1], c >> 16);
    }
  }
}

// Up to 4096 lookups: the whole sort in one workgroup, pairs handed round through LDS.
template <typename IT, int ITEMS, int BINS>
__global__ __launch_bounds__(kSortFusedThreads) void radix_sort_block_kernel(IT const *__restrict__ idx,
                                                                            uint32_t *__restrict__ keys_out,
                                                                            uint32_t *__restrict__ vals_out, int n,
                                                                            int passes, int bits, int64_t num_entries) {
  __shared__ uint32_t ks[kSortFusedThreads * ITEMS], vs[kSortFusedThreads * ITEMS];
  __shared__ uint32_t wave_off[kSortFusedWaves][BINS];
  __shared__ uint32_t wsum[BINS / 64];
  int const t = threadIdx.x, lane = t & 63, wave = t >> 6;
  int const bins = 1 << bits, mask = bins - 1;
  int const first = wave * (64 * ITEMS) + lane;
  uint32_t key[ITEMS], val[ITEMS], digit[ITEMS], rank[ITEMS];
  bool valid[ITEMS];
#pragma unroll
  for (int c = 0; c < ITEMS; c++) {
    int const i = first + c * 64;
    valid[c] = i < n;
    key[c] = valid[c] ? sort_key_at<IT, true>(idx, nullptr, i, num_entries) : 0u;
    val[c] = (uint32_t)i;
  }
  for (int pass = 0; pass < passes; pass++) {
    for (int d = lane; d < bins; d += 64) wave_off[wave][d] = 0;
#pragma unroll
    for (int c = 0; c < ITEMS; c++) digit[c] = (key[c] >> (pass * bits)) & mask;
    sort_rank_wave<ITEMS>(digit, valid, bits, lane, wave_off[wave], rank);
    __syncthreads();
    uint32_t all = 0;
    if (t < bins) {
#pragma unroll
      for (int w = 0; w < kSortFusedWaves; w++) all += wave_off[w][t];
    }
    uint32_t run = sort_scan_bins<BINS>(all, t, lane, wsum);
    if (t < bins) {
#pragma unroll
      for (int w = 0; w < kSortFusedWaves; w++) {
        uint32_t const c = wave_off[w][t];
        wave_off[w][t] = run;
        run += c;
      }
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < ITEMS; c++) {
      if (valid[c]) {
        uint32_t const pos = wave_off[wave][digit[c]] + rank[c];
        ks[pos] = key[c];
        vs[pos] = val[c];
      }
    }
    __syncthreads();
    // every key is read before the next pass's places are written: two barriers lie between
#pragma unroll
    for (int c = 0; c < ITEMS; c++) {
      if (valid[c]) {
        key[c] = ks[first + c * 64];
        val[c] = vs[first + c * 64];
      }
    }
  }
#pragma unroll
  for (int c = 0; c < ITEMS; c++) {
    if (valid[c]) {
      keys_out[first + c * 64] = key[c];
      vals_out[first + c * 64] = val[c];
    }
  }
}

struct RadixSortPlan {
  int passes;
  int bits;            // of a digit
  int ntiles;
  int items;           // fused: keys per thread
  bool fused;          // the launches below, or (one tile) one launch in all
  bool wide;           // fused: digits of up to 10 bits instead of 8
  bool scanned;        // fused: a scan launch between a pass's histogram and its scatter
  size_t table_bytes;  // fused: one [ntiles][bins] table per pass (scanned: one table and its totals); otherwise one [256][ntiles] table, then the digit totals [passes][256]
};

static inline RadixSortPlan radix_sort_plan(int64_t n, unsigned key_bits) {
  RadixSortPlan p = {};
  p.passes = (int)((key_bits + 7) / 8);
  p.bits = 8;
  // Fused while a CU each holds every tile: the table a workgroup reads grows with their number.  More
  // keys than that take the three launches a pass.
  p.fused = n <= (int64_t)kSortFusedTiles * kSortFusedThreads * kSortFusedItems;
  if (p.fused) {
    // one tile as long as four keys per thread cover everything; then as few keys per thread as the tile limit allows
    p.items = n <= kSortFusedThreads ? 1 : kSortFusedItems;
    if (n > (int64_t)kSortFusedThreads * kSortFusedItems) {
      p.items = n <= (int64_t)kSortAheadTiles * kSortFusedThreads ? 1 : n <= (int64_t)kSortFusedTiles * kSortFusedThreads * 2 ? 2 : 4;
    }
    p.ntiles = (int)ceil_div(n, (int64_t)kSortFusedThreads * p.items);
    // Digits of ten bits where they save a pass (a million rows, 20 bits: two instead of three): up to 16
    // tiles the table is still small enough for every workgroup to add up (6089 ids below 71 797 29 -> 25 us
    // with gather and walk; at 28 tiles the counts ahead cost more, 42 -> 47 us for 28 474 ids); beyond 131 072
    // lookups, where each pass has a histogram launch of its own, a third launch adds it up once (524 288 ids
    // below a million: two passes of 18-21 us instead of three of 17).  In between, neither pays.
    // (Such digits have nine or ten bits, of which the scan's workgroups take 64 at a time.)
    int const wide_passes = (int)((key_bits + 9) / 10);
    p.wide = wide_passes < p.passes && (p.ntiles <= kSortWideTiles || p.items > 1);
    if (p.wide) p.passes = wide_passes;
    p.scanned = p.wide && p.items > 1 && p.ntiles > 1;
    p.bits = (int)((key_bits + p.passes - 1) / p.passes);
    p.table_bytes = p.scanned ? ((size_t)(p.ntiles + 1) << p.bits) * sizeof(uint32_t)
                              : ((size_t)p.ntiles << p.bits) * (size_t)p.passes * sizeof(uint32_t);
  } else {
    p.ntiles = (int)ceil_div(n, kSortTile);
    p.table_bytes = (size_t)kSortRadix * ((size_t)p.ntiles + (size_t)p.passes) * sizeof(uint32_t);
  }
  return p;
}

template <typename IT, int ITEMS, int BINS>
static inline hipError_t radix_sort_fused(hipStream_t st, IT const *idx, int64_t n, int64_t num_entries,
                                          RadixSortPlan const &plan, uint32_t *keys_a, uint32_t *keys_b,
                                          uint32_t *vals_a, uint32_t *vals_b, uint32_t *table,
                                          uint32_t **keys_sorted, uint32_t **vals_sorted) {
  size_t const tsz = (size_t)plan.ntiles << plan.bits;
  unsigned const blocks = (unsigned)plan.ntiles;
  // Counting the next pass's digits while placing costs an atomic for nearly every (tile, digit)
  // pair of every workgroup: cheaper than a launch up to one key per thread, several times
  // dearer beyond (524 288 keys: 15-21 us a pass against 5 for the launch and 12 without the counting).
  constexpr bool kCountAhead = ITEMS == 1, kScanned = ITEMS > 1 && BINS > kSortRadix;
  auto tab = [&](int pass) -> uint32_t * { return pass < plan.passes ? table + (kScanned ? 0 : (size_t)pass * tsz) : nullptr; };
  auto ahead = [&](int pass) -> uint32_t * { return kCountAhead ? tab(pass) : nullptr; };
  uint32_t *kin = nullptr, *vin = nullptr, *kout = keys_a, *vout = vals_a;
  for (int pass = 0; pass < plan.passes; pass++) {
    if (pass == 0) {
      radix_hist_fused_kernel<IT, true, BINS><<<blocks, kSortFusedThreads, 0, st>>>(
          idx, nullptr, tab(0), ahead(1), n, ITEMS, 0, plan.bits, num_entries);
    } else if (!kCountAhead) {
      radix_hist_fused_kernel<IT, false, BINS><<<blocks, kSortFusedThreads, 0, st>>>(
          idx, kin, tab(pass), nullptr, n, ITEMS, plan.bits * pass, plan.bits, num_entries);
    }
    if (kScanned) {
      radix_scan_fused_kernel<<<(1u << plan.bits) / 64, kSortFusedThreads, 0, st>>>(table, table + tsz, plan.ntiles, plan.bits);
    }
    auto kern = pass == 0 ? radix_scatter_fused_kernel<IT, true, ITEMS, BINS, kScanned>
                          : radix_scatter_fused_kernel<IT, false, ITEMS, BINS, kScanned>;
    size_t const lds = ahead(pass + 1) != nullptr ? (tsz + 1) / 2 * sizeof(uint32_t) : 0;
    if (lds > (BINS > kSortRadix ? 0 : 32 * 1024)) {  // with the static part, more than a launch may ask for by default
      hipError_t const e = hipFuncSetAttribute(reinterpret_cast<void const *>(kern),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      if (e != hipSuccess) return e;
    }
    kern<<<blocks, kSortFusedThreads, lds, st>>>(idx, kin, vin, kout, vout, tab(pass), ahead(pass + 1), ahead(pass + 2), n,
                                                 plan.ntiles, plan.bits * pass, plan.bits, num_entries);
    hipError_t const e = hipGetLastError();
    if (e != hipSuccess) return e;
    kin = kout;
    vin = vout;
    kout = kin == keys_a ? keys_b : keys_a;
    vout = vin == vals_a ? vals_b : vals_a;
  }
  *keys_sorted = kin;
  *vals_sorted = vin;
  return hipSuccess;
}

// Sorts the n lookups of `idx` by row id.  bufs: two key arrays and two value
// arrays of n entries each, and the table of plan.table_bytes.  On return
// *keys_sorted / *vals_sorted point at the arrays that hold the result.
template <typename IT>
static inline hipError_t radix_sort_lookups(hipStream_t st, IT const *idx, int64_t n, int64_t num_entries,
                                            RadixSortPlan const &plan, uint32_t *keys_a, uint32_t *keys_b,
                                            uint32_t *vals_a, uint32_t *vals_b, uint32_t *table,
                                            uint32_t **keys_sorted, uint32_t **vals_sorted) {
  if (plan.fused) {
    if (plan.ntiles == 1) {
      auto kern = plan.items == 1 ? (plan.wide ? radix_sort_block_kernel<IT, 1, kSortWideRadix> : radix_sort_block_kernel<IT, 1, kSortRadix>)
                                  : (plan.wide ? radix_sort_block_kernel<IT, kSortFusedItems, kSortWideRadix>
                                               : radix_sort_block_kernel<IT, kSortFusedItems, kSortRadix>);
      kern<<<1, kSortFusedThreads, 0, st>>>(idx, keys_a, vals_a, (int)n, plan.passes, plan.bits, num_entries);
      *keys_sorted = keys_a;
      *vals_sorted = vals_a;
      return hipGetLastError();
    }
#define FFK_SORT_FUSED(ITEMS_)                                                                                      \
  return plan.wide ? radix_sort_fused<IT, ITEMS_, kSortWideRadix>(st, idx, n, num_entries, plan, keys_a, keys_b, vals_a, \
                                                                  vals_b, table, keys_sorted, vals_sorted)          \
                   : radix_sort_fused<IT, ITEMS_, kSortRadix>(st, idx, n, num_entries, plan, keys_a, keys_b, vals_a, vals_b, \
                                                              table, keys_sorted, vals_sorted)
    if (plan.items == 1) FFK_SORT_FUSED(1);
    if (plan.items == 2) FFK_SORT_FUSED(2);
    FFK_SORT_FUSED(4);
#undef FFK_SORT_FUSED
  }
  uint32_t *kin = nullptr, *vin = nullptr, *kout = keys_a, *vout = vals_a;
  uint32_t *const totals_all = table + (size_t)kSortRadix * plan.ntiles;
  radix_zero_kernel<<<plan.passes, 256, 0, st>>>(totals_all, plan.passes * kSortRadix);
  for (int pass = 0; pass < plan.passes; pass++) {
    int const shift = 8 * pass;
    unsigned const blocks = (unsigned)plan.ntiles;
    uint32_t *const totals = totals_all + pass * kSortRadix;
    if (pass == 0) {
      radix_hist_kernel<IT, true><<<blocks, kSortThreads, 0, st>>>(idx, nullptr, table, totals, n, plan.ntiles, shift, num_entries);
    } else {
      radix_hist_kernel<IT, false><<<blocks, kSortThreads, 0, st>>>(idx, kin, table, totals, n, plan.ntiles, shift, num_entries);
    }
    radix_scan_kernel<<<kSortRadix, kSortThreads, 0, st>>>(table, totals, plan.ntiles);
    if (pass == 0) {
      radix_scatter_kernel<IT, true><<<blocks, kSortThreads, 0, st>>>(idx, nullptr, nullptr, kout, vout, table, n,
                                                                     plan.ntiles, shift, num_entries);
    } else {
      radix_scatter_kernel<IT, false><<<blocks, kSortThreads, 0, st>>>(idx, kin, vin, kout, vout, table, n,
                                                                      plan.ntiles, shift, num_entries);
    }
    hipError_t const e = hipGetLastError();
    if (e != hipSuccess) return e;
    kin = kout;
    vin = vout;
    kout = kin == keys_a ? keys_b : keys_a;
    vout = vin == vals_a ? vals_b : vals_a;
  }
  *keys_sorted = kin;
  *vals_sorted = vin;
  return hipSuccess;
}

}  // namespace ffk
