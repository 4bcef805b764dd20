// Device primitives shared by the search, T-count and Clifford paths: ordered stream compaction (counts ->
// one-block scan -> scatter) and a stable LSD radix sort of (u32 key, u32 value) pairs with LDS-staged
// 8-bit digit ranking.  Kernels live in an unnamed namespace so that every translation unit has its own.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "dev.h"

namespace {
using namespace chz;

// ordered stream compaction: tiles of 256 threads x 16 items, counts -> one-block scan -> scatter
constexpr int CT_THREADS = 256, CT_ITEMS = 16, CT_TILE = CT_THREADS * CT_ITEMS;

// Kernels taking `nd` read their element count from device memory when it is not null (launches sized for a
// capacity, as in a captured graph); n is then the capacity the grid was sized for.
__device__ __forceinline__ long long dev_n(long long n, const unsigned long long *nd) {
  return nd ? (long long)*nd : n;
}

// this thread's flags of a tile: bit i for item t0 + i * CT_THREADS + thread (all items' loads in flight together)
template <typename F> __device__ __forceinline__ uint32_t tile_flags(F f, long long t0, long long n) {
  uint32_t m = 0;
#pragma unroll
  for (int i = 0; i < CT_ITEMS; i++) {
    const long long x = t0 + (long long)i * CT_THREADS + threadIdx.x;
    if (x < n && f(x)) m |= 1u << i;
  }
  return m;
}

template <typename F>
__global__ __launch_bounds__(CT_THREADS) void k_flag_count(F f, long long n, unsigned long long *bcount,
                                                           const unsigned long long *nd = nullptr) {
  n = dev_n(n, nd);
  __shared__ uint32_t ws[CT_THREADS / 64];
  const uint32_t c = gsum<64>((uint32_t)__popc(tile_flags(f, (long long)blockIdx.x * CT_TILE, n)));
  if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long s = 0;
    for (int w = 0; w < CT_THREADS / 64; w++) s += ws[w];
    bcount[blockIdx.x] = s;
  }
}

// exclusive scan of v[0..n) in place by one block; v[n] receives the total
__global__ __launch_bounds__(1024) void k_scan_one_block(unsigned long long *v, long long n) {
  __shared__ unsigned long long ws[16];
  __shared__ unsigned long long carry;
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (long long base = 0; base < n; base += 1024) {
    const long long i = base + threadIdx.x;
    const unsigned long long x = i < n ? v[i] : 0;
    unsigned long long inc = x;   // inclusive wave scan
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const unsigned long long y = __shfl_up(inc, d, 64);
      if (lane >= d) inc += y;
    }
    if (lane == 63) ws[w] = inc;
    __syncthreads();
    if (threadIdx.x == 0) {
      unsigned long long s = carry;
      for (int k = 0; k < 16; k++) { const unsigned long long t = ws[k]; ws[k] = s; s += t; }
      carry = s;
    }
    __syncthreads();
    if (i < n) v[i] = ws[w] + inc - x;
    __syncthreads();
  }
  if (threadIdx.x == 0) v[n] = carry;
}

// write(x, position) for the flagged items of the tile at t0, in order, positions from pos0; returns their number.  One
// scan over the (item, wave) counts places the whole tile: with a block scan per item, a tile's 32 barriers were most of
// a small level's compaction (15 us for 6 tiles).  The items' offsets go through LDS, so that the writes, a few items a
// thread, have their loads in flight together.
template <typename F, typename W>
__device__ __forceinline__ uint32_t tile_compact(F f, long long t0, long long n, unsigned long long pos0, W write) {
  constexpr int NW = CT_THREADS / 64;
  static_assert(CT_ITEMS * NW == 64, "the counts are scanned by one wave");
  __shared__ uint32_t ws[65];
  __shared__ uint16_t at[CT_TILE];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const uint32_t m = tile_flags(f, t0, n);
#pragma unroll
  for (int i = 0; i < CT_ITEMS; i++) {
    const uint64_t b = __ballot((m >> i) & 1u);
    if (lane == 0) ws[i * NW + w] = (uint32_t)__popcll(b);
  }
  __syncthreads();
  if (threadIdx.x < 64) {
    const uint32_t v = ws[lane];
    uint32_t inc = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t y = __shfl_up(inc, d, 64);
      if (lane >= d) inc += y;
    }
    ws[lane] = inc - v;
    if (lane == 63) ws[64] = inc;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < CT_ITEMS; i++) {
    const bool fl = (m >> i) & 1u;
    const uint64_t b = __ballot(fl);
    if (fl) at[ws[i * NW + w] + __popcll(b & ((1ull << lane) - 1))] = (uint16_t)(i * CT_THREADS + threadIdx.x);
  }
  __syncthreads();
  const uint32_t c = ws[64];
  for (uint32_t j = threadIdx.x; j < c; j += CT_THREADS) write(t0 + at[j], pos0 + j);
  return c;
}

// Sum of v[0..n) over a block of CT_THREADS threads: the tiles before a block's own, where the counts of at most
// CT_DIRECT tiles are not scanned by a launch of its own (each block reads up to 4 KB from L2; a scan and a total took
// two launches of 4 to 5 us)
constexpr long long CT_DIRECT = 512;
__device__ __forceinline__ unsigned long long tile_offset(const unsigned long long *v, long long n) {
  __shared__ uint32_t ts[CT_THREADS / 64];
  uint32_t s = 0;
  for (long long i = threadIdx.x; i < n; i += CT_THREADS) s += (uint32_t)v[i];
  s = gsum<64>(s);
  if ((threadIdx.x & 63) == 0) ts[threadIdx.x >> 6] = s;
  __syncthreads();
  unsigned long long o = 0;
  for (int w = 0; w < CT_THREADS / 64; w++) o += ts[w];
  return o;
}

// flagged positions -> ordered index list (kept survivor ranks, children needing the T bound).  boff: the tiles' offsets,
// or with tot their counts, the total then going to *tot
template <typename F>
__global__ __launch_bounds__(CT_THREADS) void k_scatter_idx(F f, long long n, const unsigned long long *boff,
                                                            uint32_t *out, const unsigned long long *nd = nullptr,
                                                            unsigned long long *tot = nullptr) {
  n = dev_n(n, nd);
  const unsigned long long pos = tot ? tile_offset(boff, blockIdx.x) : boff[blockIdx.x];
  const uint32_t c = tile_compact(f, (long long)blockIdx.x * CT_TILE, n, pos,
                                  [&](long long x, unsigned long long p) { out[p] = (uint32_t)x; });
  if (tot && threadIdx.x == 0 && blockIdx.x == gridDim.x - 1) *tot = pos + c;
}

// one tile (n <= CT_TILE) in one launch: flagged positions -> ordered index list, total written to *tot
template <typename F>
__global__ __launch_bounds__(CT_THREADS) void k_compact_one(F f, long long n, uint32_t *out, unsigned long long *tot,
                                                            const unsigned long long *nd = nullptr) {
  n = dev_n(n, nd);
  const uint32_t c = tile_compact(f, 0, n, 0, [&](long long x, unsigned long long p) { out[p] = (uint32_t)x; });
  if (threadIdx.x == 0) *tot = c;
}

// run starts (a position whose key differs from the one before and equals the one after), appended in tiles:
// each thread tests RH_ITEMS positions, a block scan places the tile's starts and one atomic per tile reserves
// their slots at *count (the runs' order does not matter: each is deduplicated on its own)
constexpr int RH_ITEMS = 16;
__attribute__((unused)) __global__ __launch_bounds__(256) void k_run_starts(const uint32_t *k, long long n,
                                                                            uint32_t *runs, unsigned long long *count,
                                                                            const unsigned long long *nd) {
  n = dev_n(n, nd);
  __shared__ unsigned long long s_wave[4], s_base;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const long long tile = 256ll * RH_ITEMS;
  for (long long t0 = (long long)blockIdx.x * tile; t0 < n; t0 += (long long)gridDim.x * tile) {
    uint32_t mask = 0;
    // (indices clamped, not branched on: all loads are in flight together)
#pragma unroll
    for (int it = 0; it < RH_ITEMS; it++) {
      const long long i = t0 + it * 256ll + tid, x = i < n ? i : n - 1;
      const uint32_t ki = k[x], kp = k[x > 0 ? x - 1 : 0], kn = k[x + 1 < n ? x + 1 : x];
      if (i < n && (i == 0 || kp != ki) && i + 1 < n && kn == ki) mask |= 1u << it;
    }
    const uint32_t c = (uint32_t)__popc(mask);
    uint32_t x = c;                                  // inclusive scan of the starts over the wave
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t y = (uint32_t)__shfl_up((int)x, d);
      if (lane >= d) x += y;
    }
    if (lane == 63) s_wave[w] = x;
    __syncthreads();
    if (tid == 0) {
      unsigned long long tot = 0;
      for (int j = 0; j < 4; j++) { const unsigned long long v = s_wave[j]; s_wave[j] = tot; tot += v; }
      s_base = tot ? atomicAdd(count, tot) : 0ull;
    }
    __syncthreads();
    unsigned long long pos = s_base + s_wave[w] + (x - c);
    for (int it = 0; it < RH_ITEMS; it++)
      if ((mask >> it) & 1u) runs[pos++] = (uint32_t)(t0 + it * 256ll + tid);
    __syncthreads();                                 // s_wave and s_base are reused by the next tile
  }
}

// ------------------------------------------------------------------------------------------------------
// Key prefixes that a sort of n survivors looks at, in passes of 8 bits: the sort only has to bring equal keys
// together, in order of their ranks, and keys that agree in a shorter prefix are told apart by the run's own comparison
// of whole keys.  At these lines a position's run holds another class with a chance of at most a quarter.
static inline int sort_passes(long long n) { return n <= (1 << 14) ? 2 : n <= (1 << 22) ? 3 : 4; }
__host__ __device__ inline uint32_t sort_prefix(uint64_t key, int passes) {
  return (uint32_t)(key >> 32) & (passes >= 4 ? 0xffffffffu : (1u << (8 * passes)) - 1);
}

// small sorts in one launch: n <= SS_MAX survivors by the low 16 bits of their prefixes, stable, two 8-bit passes in LDS
// (4096 survivors by a bitonic network of 64-bit composites: 55 us, here 11)
constexpr int SS_MAX = 4096, SS_THREADS = 1024;
__attribute__((unused)) __global__ __launch_bounds__(SS_THREADS) void k_sort_small(const uint64_t *key, long long n,
                                                                                 uint32_t *kout, uint32_t *vout,
                                                                                 const unsigned long long *nd) {
  constexpr int NW = SS_THREADS / 64;
  __shared__ uint32_t buf[2][SS_MAX];            // prefix << 12 | rank
  __shared__ uint16_t wc[NW][256];
  __shared__ uint32_t base[256], ws[4];
  n = dev_n(n, nd);
  if (n > SS_MAX) return;                  // callers take the radix sort beyond one block's LDS
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  for (int i = tid; i < n; i += SS_THREADS) buf[0][i] = sort_prefix(key[i], 2) << 12 | (uint32_t)i;
  for (int pass = 0; pass < 2; pass++) {
    const uint32_t *in = buf[pass];
    uint32_t *out = buf[pass ^ 1];
    const int shift = 12 + 8 * pass;
    if (tid < 256) base[tid] = 0;
    for (int k = tid; k < NW * 256; k += SS_THREADS) (&wc[0][0])[k] = 0;
    __syncthreads();
    for (int i = tid; i < n; i += SS_THREADS) atomicAdd(&base[(in[i] >> shift) & 255], 1u);
    __syncthreads();
    // exclusive scan of the 256 digit counts
    uint32_t inc = 0, own = 0;
    if (tid < 256) {
      own = inc = base[tid];
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const uint32_t y = __shfl_up(inc, d, 64);
        if (lane >= d) inc += y;
      }
      if (lane == 63) ws[w] = inc;
    }
    __syncthreads();
    if (tid < 256) {
      for (int k = 0; k < w; k++) inc += ws[k];
      base[tid] = inc - own;
    }
    __syncthreads();
    for (int r0 = 0; r0 < n; r0 += SS_THREADS) {
      const int i = r0 + tid;
      const bool valid = i < n;
      const uint32_t v = valid ? in[i] : 0u;
      const int dg = (int)(v >> shift) & 255;
      uint64_t peers = __ballot(valid);
#pragma unroll
      for (int b = 0; b < 8; b++) {
        const uint64_t bb = __ballot((dg >> b) & 1);
        peers &= ((dg >> b) & 1) ? bb : ~bb;
      }
      const int rank = __popcll(peers & ((1ull << lane) - 1));
      if (valid && rank == 0) wc[w][dg] = (uint16_t)__popcll(peers);
      __syncthreads();
      // the waves' counts of a digit become their start positions, the digit's base moves on
      if (tid < 256) {
        uint32_t o = base[tid];
        for (int k = 0; k < NW; k++) { const uint32_t c = wc[k][tid]; wc[k][tid] = (uint16_t)o; o += c; }
        base[tid] = o;
      }
      __syncthreads();
      if (valid) out[wc[w][dg] + rank] = v;
      __syncthreads();
      for (int k = tid; k < NW * 256; k += SS_THREADS) (&wc[0][0])[k] = 0;
      __syncthreads();
    }
  }
  for (int i = tid; i < n; i += SS_THREADS) {
    kout[i] = buf[0][i] >> 12;
    vout[i] = buf[0][i] & 0xfffu;
  }
}

// ------------------------------------------------------------------------------------------------------
// LSD radix sort of (u32 key, u32 value) pairs, 8-bit digits, stable: tiles of 1024 threads x 2 rounds.  (With 256 threads
// x 8 rounds a tile's scatter was a chain of 24 barriers, which is what a sort of a few tiles takes: 12 us, here 7.)
constexpr int RS_THREADS = 1024, RS_ROUNDS = 2, RS_TILE = RS_THREADS * RS_ROUNDS;

// counts of this tile's digits in h (256, shared)
__device__ __forceinline__ void radix_tile_counts(const uint32_t *keys, long long n, int shift, unsigned int *h) {
  if (threadIdx.x < 256) h[threadIdx.x] = 0;
  __syncthreads();
  const long long t0 = (long long)blockIdx.x * RS_TILE;
#pragma unroll
  for (int r = 0; r < RS_ROUNDS; r++) {
    const long long x = t0 + (long long)r * RS_THREADS + threadIdx.x;
    if (x < n) atomicAdd(&h[(keys[x] >> shift) & 255], 1u);
  }
  __syncthreads();
}

__global__ __launch_bounds__(RS_THREADS) void k_radix_hist(const uint32_t *keys, long long n, int shift,
                                                           unsigned long long *hist, long long nblocks,
                                                           const unsigned long long *nd = nullptr) {
  n = dev_n(n, nd);
  __shared__ unsigned int h[256];
  radix_tile_counts(keys, n, shift, h);
  if (threadIdx.x < 256) hist[(long long)threadIdx.x * nblocks + blockIdx.x] = h[threadIdx.x];
}

// this block's tile of (key, value) pairs placed from base[d], the first output position of digit d for the tile
// (shared)
__device__ __forceinline__ void radix_scatter_tile(const uint32_t *kin, const uint32_t *vin, long long n, int shift,
                                                   unsigned long long *base, uint32_t *kout, uint32_t *vout) {
  constexpr int NW = RS_THREADS / 64;
  __shared__ uint16_t wc[RS_ROUNDS][NW][256];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  for (int k = tid; k < RS_ROUNDS * NW * 128; k += RS_THREADS) ((uint32_t *)wc)[k] = 0;
  const long long t0 = (long long)blockIdx.x * RS_TILE;
  uint32_t key[RS_ROUNDS], val[RS_ROUNDS];
  int rank[RS_ROUNDS];
#pragma unroll
  for (int r = 0; r < RS_ROUNDS; r++) {
    const long long x = t0 + (long long)r * RS_THREADS + tid;
    key[r] = x < n ? kin[x] : 0u;
    val[r] = x < n ? vin[x] : 0u;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < RS_ROUNDS; r++) {
    const bool valid = t0 + (long long)r * RS_THREADS + tid < n;
    const int dg = (key[r] >> shift) & 255;
    uint64_t peers = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; b++) {
      const uint64_t bb = __ballot((dg >> b) & 1);
      peers &= ((dg >> b) & 1) ? bb : ~bb;
    }
    rank[r] = __popcll(peers & ((1ull << lane) - 1));
    if (valid && rank[r] == 0) wc[r][w][dg] = (uint16_t)__popcll(peers);
  }
  __syncthreads();
  // the (round, wave) counts of a digit become offsets from its base
  if (tid < 256) {
    uint32_t o = 0;
    for (int k = 0; k < RS_ROUNDS * NW; k++) {
      uint16_t &c = (&wc[0][0][0])[k * 256 + tid];
      const uint32_t v = c;
      c = (uint16_t)o;
      o += v;
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < RS_ROUNDS; r++) {
    if (t0 + (long long)r * RS_THREADS + tid >= n) continue;
    const int dg = (key[r] >> shift) & 255;
    const unsigned long long p = base[dg] + wc[r][w][dg] + rank[r];
    kout[p] = key[r];
    vout[p] = val[r];
  }
}

__global__ __launch_bounds__(RS_THREADS) void k_radix_scatter(const uint32_t *kin, const uint32_t *vin, long long n,
                                                              int shift, const unsigned long long *hist,
                                                              long long nblocks, uint32_t *kout, uint32_t *vout,
                                                              const unsigned long long *nd = nullptr) {
  n = dev_n(n, nd);
  __shared__ unsigned long long base[256];
  if (threadIdx.x < 256) base[threadIdx.x] = hist[(long long)threadIdx.x * nblocks + blockIdx.x];
  radix_scatter_tile(kin, vin, n, shift, base, kout, vout);
}

// Sorts of up to RS_DIRECT_MAX tiles skip the scan of the histogram: k_radix_count writes each tile's digit counts
// (cnt[tile * 256 + d], 32-bit) and every scatter block forms its own 256 start positions from them, the counts of
// all smaller digits plus those of its digit in earlier tiles.  Two launches per pass instead of six (count, three
// scan kernels, the scan's total, scatter); each block reads the whole count table, at most 512 KB from L2.
constexpr long long RS_DIRECT_MAX = 512;

__global__ __launch_bounds__(RS_THREADS) void k_radix_count(const uint32_t *keys, long long n, int shift,
                                                            uint32_t *cnt, const unsigned long long *nd = nullptr) {
  n = dev_n(n, nd);
  __shared__ unsigned int h[256];
  radix_tile_counts(keys, n, shift, h);
  if (threadIdx.x < 256) cnt[(long long)blockIdx.x * 256 + threadIdx.x] = h[threadIdx.x];
}

__global__ __launch_bounds__(RS_THREADS) void k_radix_scatter_direct(const uint32_t *kin, const uint32_t *vin,
                                                                     long long n, int shift, const uint32_t *cnt,
                                                                     long long nblocks, uint32_t *kout,
                                                                     uint32_t *vout,
                                                                     const unsigned long long *nd = nullptr) {
  n = dev_n(n, nd);
  // the tiles that hold no element place nothing (launches sized for a capacity)
  if ((long long)blockIdx.x * RS_TILE >= n) return;
  const long long used = (n + RS_TILE - 1) / RS_TILE;
  if (used < nblocks) nblocks = used;
  constexpr int Q = RS_THREADS / 256;
  __shared__ unsigned long long base[256];
  __shared__ uint32_t stot[Q][256], sbel[Q][256];
  __shared__ uint32_t wsum[4];
  const int d = threadIdx.x & 255, qq = threadIdx.x >> 8, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  // digit d: its count over all tiles and over the tiles before this one (coalesced rows of 256 counts), every Q-th tile
  uint32_t tot = 0, below = 0;
  const long long me = blockIdx.x;
#pragma unroll 4
  for (long long t = qq; t < nblocks; t += Q) {
    const uint32_t c = cnt[t * 256 + d];
    tot += c;
    below += t < me ? c : 0u;
  }
  stot[qq][d] = tot;
  sbel[qq][d] = below;
  __syncthreads();
  // exclusive scan of the digit totals over the 256 digits
  uint32_t inc = 0;
  if (threadIdx.x < 256) {
    tot = below = 0;
    for (int k = 0; k < Q; k++) { tot += stot[k][d]; below += sbel[k][d]; }
    inc = tot;
#pragma unroll
    for (int k = 1; k < 64; k <<= 1) {
      const uint32_t y = __shfl_up(inc, k, 64);
      if (lane >= k) inc += y;
    }
    if (lane == 63) wsum[w] = inc;
  }
  __syncthreads();
  if (threadIdx.x < 256) {
    uint32_t off = 0;
    for (int k = 0; k < w; k++) off += wsum[k];
    base[d] = (unsigned long long)off + inc - tot + below;
  }
  radix_scatter_tile(kin, vin, n, shift, base, kout, vout);     // (its first barrier orders base)
}


// ------------------------------------------------------------------------------------------------------
// exclusive scan of long arrays: tiles of 4096 entries scanned in place, tile totals scanned by one block,
// tile offsets added back
constexpr int SC_THREADS = 1024, SC_ITEMS = 4, SC_TILE = SC_THREADS * SC_ITEMS;

__global__ __launch_bounds__(SC_THREADS) void k_scan_tiles(unsigned long long *v, long long n,
                                                          unsigned long long *tot) {
  __shared__ unsigned long long ws[SC_THREADS / 64];
  const long long base = (long long)blockIdx.x * SC_TILE + (long long)threadIdx.x * SC_ITEMS;
  unsigned long long x[SC_ITEMS], s = 0;
#pragma unroll
  for (int i = 0; i < SC_ITEMS; i++) { x[i] = base + i < n ? v[base + i] : 0; s += x[i]; }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  unsigned long long inc = s;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const unsigned long long y = __shfl_up(inc, d, 64);
    if (lane >= d) inc += y;
  }
  if (lane == 63) ws[w] = inc;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long a = 0;
    for (int k = 0; k < SC_THREADS / 64; k++) { const unsigned long long t = ws[k]; ws[k] = a; a += t; }
    tot[blockIdx.x] = a;
  }
  __syncthreads();
  unsigned long long e = ws[w] + inc - s;
#pragma unroll
  for (int i = 0; i < SC_ITEMS; i++) {
    if (base + i < n) v[base + i] = e;
    e += x[i];
  }
}

__global__ void k_scan_add(unsigned long long *v, long long n, const unsigned long long *tot) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    v[i] += tot[i / SC_TILE];
}

// v[0..n) <- exclusive prefix sums, v[n] <- total.  tmp holds at least n / SC_TILE + 2 entries.
static inline hipError_t scan_excl(unsigned long long *v, long long n, unsigned long long *tmp, hipStream_t s) {
  if (n <= 4 * SC_TILE) {
    hipLaunchKernelGGL(k_scan_one_block, dim3(1), dim3(1024), 0, s, v, n);
    return hipGetLastError();
  }
  const long long nt = (n + SC_TILE - 1) / SC_TILE;
  hipLaunchKernelGGL(k_scan_tiles, dim3((unsigned)nt), dim3(SC_THREADS), 0, s, v, n, tmp);
  hipLaunchKernelGGL(k_scan_one_block, dim3(1), dim3(1024), 0, s, tmp, nt);
  hipLaunchKernelGGL(k_scan_add, dim3((unsigned)std::min<long long>((n + 255) / 256, 16384)), dim3(256), 0, s, v, n,
                     tmp);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  return hipMemcpyAsync(v + n, tmp + nt, sizeof(unsigned long long), hipMemcpyDeviceToDevice, s);
}

// stable sort of n (u32 key, u32 value) pairs by the low 8 * passes bits: (k0, v0) -> (k0, v0) through (k1, v1); an odd
// number of passes starts from (k1, v1).
// hist holds at least 256 * ceil(n / RS_TILE) + 1 entries, tmp what scan_excl needs for that many.
// With nd the count is read on the device and n is the capacity the launches are sized for.
static inline hipError_t radix_sort_pairs(uint32_t *k0, uint32_t *v0, uint32_t *k1, uint32_t *v1, long long n,
                                          unsigned long long *hist, unsigned long long *tmp, hipStream_t s,
                                          const unsigned long long *nd = nullptr, int passes = 4) {
  if (n < 1 || (n == 1 && passes % 2 == 0)) return hipSuccess;
  const long long nb = (n + RS_TILE - 1) / RS_TILE;
  uint32_t *ks[2] = {k0, k1}, *vs[2] = {v0, v1};
  if (nb <= RS_DIRECT_MAX) {
    uint32_t *cnt = reinterpret_cast<uint32_t *>(hist);     // nb * 256 counts fit the histogram's space
    for (int pass = 0; pass < passes; pass++) {
      const int a = (pass + passes) & 1, b = a ^ 1;
      hipLaunchKernelGGL(k_radix_count, dim3((unsigned)nb), dim3(RS_THREADS), 0, s, ks[a], n, pass * 8, cnt, nd);
      hipLaunchKernelGGL(k_radix_scatter_direct, dim3((unsigned)nb), dim3(RS_THREADS), 0, s, ks[a], vs[a], n,
                         pass * 8, cnt, nb, ks[b], vs[b], nd);
    }
    return hipGetLastError();
  }
  for (int pass = 0; pass < passes; pass++) {
    const int a = (pass + passes) & 1, b = a ^ 1;
    hipLaunchKernelGGL(k_radix_hist, dim3((unsigned)nb), dim3(RS_THREADS), 0, s, ks[a], n, pass * 8, hist, nb, nd);
    hipError_t e = scan_excl(hist, nb * 256, tmp, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_radix_scatter, dim3((unsigned)nb), dim3(RS_THREADS), 0, s, ks[a], vs[a], n, pass * 8, hist,
                       nb, ks[b], vs[b], nd);
  }
  return hipGetLastError();
}

}  // namespace
