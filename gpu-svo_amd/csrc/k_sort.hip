// k_sort.hip -- LSD radix sort of voxel keys: 8-bit digits, three kernels per
// digit pass (reduce, scan, scatter).
//
// Replaces the reference's dense flag array + exclusive scan + compaction
// (SVO.cu:367-405), which is O(res^3), with a sort of the emitted hit keys,
// O(hits).  The sorted order equals the reference's index order of the dense
// array (keys are the Morton codes).
//
// The key count n is read from device memory, so no launch shape depends on
// the hit count.  Kernels of a pass:
//   k_tile_hist   digit counts of each tile, stored digit-major
//   k_tile_scan   per digit, exclusive scan over the tiles and the total
//   k_scatter     the digits' offsets from the totals; ranks the tile's keys
//                 stably with wave64 match masks (8 ballots per 64 keys) and
//                 writes them through an LDS reorder so the stores are
//                 contiguous within each digit run
// Stable, so the passes compose into a full LSD sort.  HBM traffic for n keys
// of B bytes and P passes: P * 3*n*B, plus 2 KB of counts per tile and pass.
// A single-pass scatter with decoupled look-back reads and writes the keys
// once per pass, but over thousands of tiles its look-back chain (and the
// digits' status words each tile walks) bounds the pass; here no tile waits on
// another.
//
// A pass of a million 4-byte keys costs 16 us, 10 of it the three launches
// (83 -> 68 us for 30 bits since the digits' offsets come from the passes' own
// counts: one read of the keys for all digit histograms and its two small
// launches cost more).  Digits of 9 and 10 bits, which save a pass of four or
// five, were slower from 300,000 keys on (10 bits: 89 us against 68 at a
// million, 243 against 146 at four) and no better than 1 us below.
#include <algorithm>
#include <utility>

#include "svo_internal.h"
#include "svo_scan.h"

namespace svo {
namespace {

constexpr int BLOCK = 256;
constexpr int WAVES = BLOCK / 64;
constexpr int DIGIT = 8, RADIX = 1 << DIGIT;
static_assert(RADIX == BLOCK, "a thread per digit");
// Keys per lane and tile: fewer for fewer keys, so that small sorts have
// workgroups for the 256 CUs.  30-bit keys of 4 bytes, 4 / 8 / 16 keys a lane:
// 100,000 keys 47 / 54 / 60 us, a million 78 / 68 / 71, four million
// 193 / 146 / 125.  The size is chosen by `cap`, which is the number of keys at
// the library's sort entry points; a build's pass knows its candidate cells
// only, 5.5 times its keys where triangles are large (4.95 of 27.45 million on
// 150,000 triangles at 4096^3), so that its tiles are those of a larger sort.
constexpr uint64_t TINY_SORT = 1ull << 18, SMALL_SORT = 1ull << 21;
constexpr int KPT_TINY = 4, KPT_SMALL = 8, KPT_LARGE = 16;

struct SortPlan {
  int passes, kpt;
  uint64_t tile, tiles;
};
SortPlan sort_plan(uint64_t cap, int bits) {
  SortPlan p;
  cap = std::max<uint64_t>(cap, 1);
  p.passes = (bits + DIGIT - 1) / DIGIT;
  p.kpt = cap < TINY_SORT ? KPT_TINY : cap < SMALL_SORT ? KPT_SMALL : KPT_LARGE;
  p.tile = (uint64_t)BLOCK * p.kpt;
  p.tiles = (cap + p.tile - 1) / p.tile;
  return p;
}

// Digit counts of tiles blockIdx.x, + gridDim.x, ...: counts[d * tiles + t].
// With `copy`, the keys are written there as well.
template <typename K, int KPT>
__global__ __launch_bounds__(BLOCK) void k_tile_hist(const K* in, const unsigned long long* n_ptr,
                                                     int shift, uint32_t dm, uint32_t* counts,
                                                     uint64_t tiles, K* copy) {
  constexpr int TILE = BLOCK * KPT;
  __shared__ uint32_t h[WAVES][RADIX];
  const uint32_t w = threadIdx.x >> 6;
  const uint64_t n = *n_ptr;
  const uint64_t n_tiles = (n + TILE - 1) / TILE;
  const bool vec = ((uintptr_t)in & 15) == 0;
  for (uint64_t tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
    for (int i = __lane_id(); i < RADIX; i += 64) h[w][i] = 0;
    __syncthreads();
    // thread: KPT consecutive keys of the tile; runs of equal digits are
    // added at once
    const uint64_t b = tile * TILE + (uint64_t)threadIdx.x * KPT;
    const uint32_t cnt = b < n ? (uint32_t)((n - b) < KPT ? (n - b) : KPT) : 0u;
    K kk[KPT];
    load_consecutive(in + (b < n ? b : 0), vec && b < n, cnt, kk);
    if (copy)
#pragma unroll
      for (int j = 0; j < KPT; ++j)
        if ((uint32_t)j < cnt) copy[b + j] = kk[j];
    if (cnt) {
      uint32_t last = (uint32_t)(kk[0] >> shift) & dm, run = 1;
#pragma unroll
      for (int j = 1; j < KPT; ++j) {
        if ((uint32_t)j < cnt) {
          const uint32_t d = (uint32_t)(kk[j] >> shift) & dm;
          if (d == last) {
            ++run;
          } else {
            atomicAdd(&h[w][last], run);
            last = d;
            run = 1;
          }
        }
      }
      atomicAdd(&h[w][last], run);
    }
    __syncthreads();
    {
      const uint32_t d = threadIdx.x;
      uint32_t c = 0;
#pragma unroll
      for (int k = 0; k < WAVES; ++k) c += h[k][d];
      counts[(uint64_t)d * tiles + tile] = c;
    }
    __syncthreads();
  }
}

// Block d: exclusive scan of counts[d * tiles + 0 .. n_tiles) in place; their
// sum to totals[d].
__global__ __launch_bounds__(BLOCK) void k_tile_scan(uint32_t* counts,
                                                     const unsigned long long* n_ptr,
                                                     uint64_t tiles, uint64_t tile, uint32_t* totals) {
  __shared__ uint32_t tmp[4];
  const uint64_t n_tiles = (*n_ptr + tile - 1) / tile;
  uint32_t* c = counts + (uint64_t)blockIdx.x * tiles;
  uint32_t run = 0;
  constexpr int PER = 16;
  for (uint64_t t0 = 0; t0 < n_tiles; t0 += (uint64_t)BLOCK * PER) {
    const uint64_t i0 = t0 + (uint64_t)threadIdx.x * PER;
    uint32_t v[PER], sum = 0;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      v[j] = i0 + j < n_tiles ? c[i0 + j] : 0u;
      sum += v[j];
    }
    uint32_t total;
    uint32_t p = run + block_excl_scan256(sum, tmp, total);
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      if (i0 + j < n_tiles) c[i0 + j] = p;
      p += v[j];
    }
    run += total;
    __syncthreads();  // tmp is reused by the next chunk's scan
  }
  if (threadIdx.x == 0) totals[blockIdx.x] = run;
}

// One digit pass over tiles blockIdx.x, + gridDim.x, ...: the tile's keys
// are ranked stably, reordered in LDS by digit and written to where
// k_tile_scan put the tile's run of each digit.
template <typename K, int KPT>
__global__ __launch_bounds__(BLOCK) void k_scatter(const K* in, K* out,
                                                   const unsigned long long* n_ptr, int shift,
                                                   uint32_t dm, const uint32_t* starts,
                                                   const uint32_t* totals, uint64_t tiles) {
  constexpr int TILE = BLOCK * KPT;
  __shared__ uint32_t wcnt[WAVES][RADIX];
  __shared__ uint32_t dbase[RADIX];
  __shared__ uint32_t tstart[RADIX];
  __shared__ uint32_t tmp[4];
  __shared__ K sorted[TILE];
  const uint32_t w = threadIdx.x >> 6;
  const uint32_t lane = __lane_id();
  const uint64_t n = *n_ptr;
  const uint64_t n_tiles = (n + TILE - 1) / TILE;
  if (blockIdx.x >= n_tiles) return;
  uint32_t total;
  const uint32_t first = block_excl_scan256(totals[threadIdx.x], tmp, total);
  for (uint64_t tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
    for (int i = lane; i < RADIX; i += 64) wcnt[w][i] = 0;
    dbase[threadIdx.x] = first + starts[(uint64_t)threadIdx.x * tiles + tile];
    __syncthreads();
    const uint64_t tb = tile * TILE;
    const uint32_t tn = (uint32_t)((n - tb) < TILE ? (n - tb) : TILE);
    // loads first, all in flight together (indices clamped, so unconditional)
    K keys[KPT];
#pragma unroll
    for (int it = 0; it < KPT; ++it) {
      const uint32_t pos = w * (KPT * 64) + it * 64 + lane;
      const K v = in[tb + (pos < tn ? pos : tn - 1)];
      keys[it] = pos < tn ? v : (K)0;
    }
    // stable rank within the wave: match masks per 64 keys; the group leader
    // reserves the group's slots in the wave's digit counter (LDS atomics
    // return the old counts; the 16 reservations are waited on together)
    uint32_t rank[KPT], lead[KPT], base[KPT];
#pragma unroll
    for (int it = 0; it < KPT; ++it) {
      const uint32_t pos = w * (KPT * 64) + it * 64 + lane;
      const bool valid = pos < tn;
      const uint32_t d = (uint32_t)(keys[it] >> shift) & dm;
      uint64_t eq = __ballot(valid);
#pragma unroll
      for (int bit = 0; bit < DIGIT; ++bit) {
        // lanes whose bit equals this lane's: ~(ballot ^ (bit ? ~0 : 0))
        const uint32_t sx = (uint32_t)((int32_t)(d << (31 - bit)) >> 31);
        const uint64_t m = __ballot(sx != 0);
        eq &= ~(m ^ (((uint64_t)sx << 32) | sx));
      }
      lead[it] = valid ? (uint32_t)__builtin_ctzll(eq) : 0u;
      rank[it] = lanes_below(eq);
      base[it] = 0;
      if (valid && lane == lead[it]) base[it] = atomicAdd(&wcnt[w][d], (uint32_t)__popcll(eq));
    }
#pragma unroll
    for (int it = 0; it < KPT; ++it) rank[it] += __shfl(base[it], (int)lead[it]);
    __syncthreads();
    {
      const uint32_t d = threadIdx.x;
      uint32_t cnt = 0;
#pragma unroll
      for (int k = 0; k < WAVES; ++k) {
        const uint32_t c = wcnt[k][d];
        wcnt[k][d] = cnt;
        cnt += c;
      }
      tstart[d] = block_excl_scan256(cnt, tmp, total);
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < KPT; ++it) {
      const uint32_t pos = w * (KPT * 64) + it * 64 + lane;
      if (pos < tn) {
        const uint32_t d = (uint32_t)(keys[it] >> shift) & dm;
        sorted[tstart[d] + wcnt[w][d] + rank[it]] = keys[it];
      }
    }
    __syncthreads();
    // write out in tile order: consecutive threads store consecutive keys of
    // a digit run
    K sk[KPT];
#pragma unroll
    for (int it = 0; it < KPT; ++it) {
      const uint32_t i = it * BLOCK + threadIdx.x;
      sk[it] = sorted[i < tn ? i : 0];
    }
#pragma unroll
    for (int it = 0; it < KPT; ++it) {
      const uint32_t i = it * BLOCK + threadIdx.x;
      const uint32_t d = (uint32_t)(sk[it] >> shift) & dm;
      const uint64_t o = (uint64_t)dbase[d] + (i - tstart[d]);
      if (i < tn) out[o] = sk[it];
    }
    __syncthreads();
  }
}

}  // namespace

size_t radix_sort_tmp_bytes(uint64_t cap) {
  return (size_t)(sort_plan(cap, 0).tiles + 1) * RADIX * sizeof(uint32_t) + 256;
}
size_t radix_sort_tmp_bound(uint64_t cap) {
  return std::max({radix_sort_tmp_bytes(std::min(cap, TINY_SORT - 1)),
                   radix_sort_tmp_bytes(std::min(cap, SMALL_SORT - 1)), radix_sort_tmp_bytes(cap)});
}

namespace {
template <typename K, int KPT>
void sort_passes(const SortPlan& p, K* src, K* dst, K* copy, const unsigned long long* n, int bits,
                 uint32_t grid, void* tmp, hipStream_t s) {
  uint32_t* counts = (uint32_t*)tmp;
  uint32_t* totals = counts + p.tiles * RADIX;
  for (int i = 0; i < p.passes; ++i) {
    const int shift = DIGIT * i;
    const uint32_t dm = (1u << std::min(DIGIT, bits - shift)) - 1u;
    hipLaunchKernelGGL((k_tile_hist<K, KPT>), dim3(grid), dim3(BLOCK), 0, s, (const K*)src, n,
                       shift, dm, counts, p.tiles, copy);
    if (copy) {
      std::swap(src, dst);
      copy = nullptr;
    }
    hipLaunchKernelGGL(k_tile_scan, dim3(RADIX), dim3(BLOCK), 0, s, counts, n, p.tiles, p.tile,
                       totals);
    hipLaunchKernelGGL((k_scatter<K, KPT>), dim3(grid), dim3(BLOCK), 0, s, (const K*)src, dst,
                       n, shift, dm, (const uint32_t*)counts, (const uint32_t*)totals, p.tiles);
    std::swap(src, dst);
  }
}
}  // namespace

template <typename K>
void launch_radix_sort(K* a, K* b, const unsigned long long* n, uint64_t cap, int bits,
                       uint32_t blocks, void* tmp, K** result, hipStream_t s) {
  const SortPlan p = sort_plan(cap, bits);
  // tiles are independent: at most `blocks` workgroups, each taking tiles
  // blockIdx.x, + gridDim.x, ...
  const uint32_t grid = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(p.tiles, blocks));
  // without `result` the keys end in a: an odd number of passes starts from
  // a copy in b, which the first pass's counting makes
  K* copy = !result && (p.passes & 1) ? b : nullptr;
  if (p.kpt == KPT_TINY) sort_passes<K, KPT_TINY>(p, a, b, copy, n, bits, grid, tmp, s);
  else if (p.kpt == KPT_SMALL) sort_passes<K, KPT_SMALL>(p, a, b, copy, n, bits, grid, tmp, s);
  else sort_passes<K, KPT_LARGE>(p, a, b, copy, n, bits, grid, tmp, s);
  if (result) *result = (p.passes & 1) ? b : a;
}

template void launch_radix_sort<uint32_t>(uint32_t*, uint32_t*, const unsigned long long*,
                                          uint64_t, int, uint32_t, void*, uint32_t**,
                                          hipStream_t);
template void launch_radix_sort<uint64_t>(uint64_t*, uint64_t*, const unsigned long long*,
                                          uint64_t, int, uint32_t, void*, uint64_t**,
                                          hipStream_t);

}  // namespace svo
