// k_levels.hip -- sorted unique voxels and the bottom-up octree levels.
//
// Reference: the level loop of SparseVoxelOctree::create (SVO.cu:383-495).
// Per level it flags parent-group heads (cpNumNodes, SVO.cu:221-235), scans
// them (SVO.cu:433-437), places node i at sum[i] + (code & 7) (createNode_*,
// SVO.cu:237-309), fills the empty siblings (createRemainNode, 311-339) and
// stops at the first level holding a single code (487-490).
//
// Here every level is one pass over the level's sorted unique keys:
//   group head  = first key of its parent group (parent differs from the
//                 previous key's parent; composite keys keep meshes apart),
//   root        = the only key of its mesh at this level (the reference's
//                 single-code level), which ends that mesh's tree,
//   output      = next level's keys (the group parents, already sorted and
//                 unique) and, per group, the index of its first child and the
//                 mask of the children it has.
// Level 1 is fused with the de-duplication of the sorted hit keys.  Node
// records are written later from these arrays (k_attrs.hip), once the node
// counts are known.
//
// Each pass is a single-pass scan: workgroups claim tiles by ticket, each
// thread loads consecutive keys with vector loads, the tile's counts are
// scanned in the workgroup and its offset found by decoupled look-back
// (svo_scan.h); compacted outputs are staged in LDS and written contiguously.
// The element count is read from device memory, so no launch shape depends on
// it.  The coarse levels, a few thousand elements at most, run in one
// workgroup and one launch together.
#include <algorithm>

#include "svo_internal.h"
#include "svo_scan.h"

namespace svo {
namespace {

constexpr int BLOCK = 256;
constexpr int EPT = 16;             // consecutive elements per thread
constexpr int TILE = BLOCK * EPT;   // 4096
constexpr int MAX_TICKETS = 64;     // one per pass: level 1 .. level 63
// Level passes over fewer elements than fill the chip with 4096-element tiles
// take 1024-element tiles (4 per thread).
constexpr int EPT_SMALL = 4, TILE_SMALL = BLOCK * EPT_SMALL;
constexpr uint64_t SMALL_ELEMS = 256 * TILE;

// Tiles, at most, of a level pass over up to n elements.
__host__ __device__ inline uint64_t level_tiles(uint64_t n) {
  const uint64_t big = (n + TILE - 1) / TILE;
  const uint64_t m = n < SMALL_ELEMS ? n : SMALL_ELEMS;
  const uint64_t small = (m + TILE_SMALL - 1) / TILE_SMALL;
  return big > small ? big : small;
}

// flags of sorted hit key `cur`: bit0 = first copy of its key, bit1 = head of
// its parent group
template <typename K>
__device__ inline uint32_t first_flags_v(K prev, K cur, bool has_prev, KeyLayout<K> kl) {
  if (!has_prev) return 3u;
  if (cur == prev) return 0u;
  return 1u | (kl.parent(cur) != kl.parent(prev) ? 2u : 0u);
}

// flags of level element `cur` of a mesh still being built: bit1 = group
// head, bit2 = the only element of its mesh (the root)
template <typename K>
__device__ inline uint32_t level_flags_v(K prev, K cur, K next, bool has_prev, bool has_next,
                                         KeyLayout<K> kl) {
  const uint32_t m = kl.mesh(cur);
  const bool first = !has_prev || kl.mesh(prev) != m;
  const bool last = !has_next || kl.mesh(next) != m;
  if (first && last) return 4u;
  if (first) return 2u;
  return kl.parent(cur) != kl.parent(prev) ? 2u : 0u;
}

__global__ __launch_bounds__(BLOCK) void k_level_clear(uint64_t* status, uint32_t* tickets,
                                                       const unsigned long long* n_ptr) {
  const uint64_t words = 2 * level_tiles(*n_ptr);
  const uint64_t stride = (uint64_t)gridDim.x * BLOCK;
  for (uint64_t i = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; i < words; i += stride)
    status[i] = 0;
  if (blockIdx.x == 0 && threadIdx.x < MAX_TICKETS) tickets[threadIdx.x] = 0;
}

// Per-tile frame shared by both passes: claims a tile, loads the thread's run
// and the keys just before and after it.
template <typename K>
struct TileRun {
  uint64_t tile, tb, i0;
  uint32_t tn, cnt;
  K kk[EPT];
  K prev, next;
  bool has_prev, has_next;
};

template <typename K>
__device__ inline bool claim_tile(const K* src, uint64_t n, uint32_t* ticket, uint32_t* s_tile,
                                  K (*s_edge)[BLOCK], TileRun<K>& r) {
  if (threadIdx.x == 0) *s_tile = atomicAdd(ticket, 1u);
  __syncthreads();
  r.tile = *s_tile;
  r.tb = r.tile * TILE;
  if (r.tb >= n) return false;  // uniform over the workgroup
  r.tn = (uint32_t)((n - r.tb) < TILE ? (n - r.tb) : TILE);
  const uint32_t l0 = threadIdx.x * EPT;
  r.cnt = l0 < r.tn ? ((r.tn - l0) < EPT ? (r.tn - l0) : EPT) : 0u;
  r.i0 = r.tb + l0;
  load_consecutive(src + r.i0, ((uintptr_t)src & 15) == 0, r.cnt, r.kk);
  K last = r.kk[0];
#pragma unroll
  for (int e = 1; e < EPT; ++e)
    if ((uint32_t)e < r.cnt) last = r.kk[e];
  s_edge[0][threadIdx.x] = r.kk[0];
  s_edge[1][threadIdx.x] = last;
  __syncthreads();
  r.has_prev = r.cnt && r.i0 > 0;
  r.prev = !r.has_prev ? (K)0 : threadIdx.x > 0 ? s_edge[1][threadIdx.x - 1] : src[r.i0 - 1];
  r.has_next = r.cnt && r.i0 + r.cnt < n;
  r.next = !r.has_next ? (K)0
           : (threadIdx.x + 1 < BLOCK && l0 + EPT < r.tn) ? s_edge[0][threadIdx.x + 1]
                                                           : src[r.i0 + r.cnt];
  return true;
}

// ---------------------------------------------------------------- level 1
// Sorted hit keys -> unique keys (elem1), the level-2 keys (elem2 = group
// parents) with their first child (first_child2), the per-mesh spans of
// level 1, and counts[0] / counts[1].  (Level 1's own group index per key is
// not needed: node records look groups up from the level above.)
template <typename K>
__global__ __launch_bounds__(BLOCK) void k_first_pass(
    const K* sorted, const unsigned long long* n_ptr, KeyLayout<K> kl, K* elem1, K* elem2,
    uint32_t* first_child2, LevelSpan* spans, uint32_t n_levels,
    uint64_t* status, uint32_t* ticket, uint32_t epoch, unsigned long long* counts) {
  __shared__ K s_edge[2][BLOCK];
  __shared__ K s_key[TILE];
  __shared__ uint32_t s_val[TILE];
  __shared__ uint64_t tmp[4];
  __shared__ uint32_t s_tile;
  __shared__ uint32_t s_base[2];
  const uint64_t n = *n_ptr;
  TileRun<K> r;
  while (claim_tile(sorted, n, ticket, &s_tile, s_edge, r)) {
    uint32_t f = 0, nu = 0, ng = 0;
    {
      K pk = r.prev;
      bool hp = r.has_prev;
#pragma unroll
      for (int e = 0; e < EPT; ++e) {
        if ((uint32_t)e < r.cnt) {
          const uint32_t fl = first_flags_v(pk, r.kk[e], hp, kl);
          f |= fl << (2 * e);
          nu += fl & 1u;
          ng += fl >> 1;
          pk = r.kk[e];
          hp = true;
        }
      }
    }
    uint64_t tot;
    const uint64_t ex = block_excl_scan256(((uint64_t)ng << 32) | nu, tmp, tot);
    const uint32_t tu = (uint32_t)tot, tg = (uint32_t)(tot >> 32);
    if (threadIdx.x < 128) {
      // wave 0: unique-key offset, wave 1: group offset
      const uint32_t wv = threadIdx.x >> 6;
      const uint32_t c = wv == 0 ? tu : tg;
      const uint32_t pre = lookback_exclusive_wave(status + wv, 2, r.tile, c, epoch);
      if (__lane_id() == 0) {
        s_base[wv] = pre;
        if (r.tb + r.tn == n) counts[wv] = (unsigned long long)pre + c;
      }
    }
    __syncthreads();
    const uint32_t bu = s_base[0], bg = s_base[1];
    // elem1 staged by tile-local unique index; spans on the way
    {
      uint32_t ru = (uint32_t)ex, rg = (uint32_t)(ex >> 32);
      K pk = r.prev;
      bool hp = r.has_prev;
#pragma unroll
      for (int e = 0; e < EPT; ++e) {
        if ((uint32_t)e < r.cnt) {
          const K key = r.kk[e];
          const uint32_t fl = (f >> (2 * e)) & 3u;
          const uint32_t m = kl.mesh(key);
          if (fl & 1u) {
            if (fl & 2u) ++rg;
            s_key[ru] = key;
            if (!hp || kl.mesh(pk) != m) {  // first element of its mesh
              spans[(uint64_t)m * n_levels].elem_first = bu + ru;
              spans[(uint64_t)m * n_levels].group_first = bg + rg - 1;
            }
            ++ru;
          }
          const bool hn = (uint32_t)e + 1 < r.cnt || r.has_next;
          const K nk = (uint32_t)e + 1 < r.cnt ? r.kk[e + 1 < EPT ? e + 1 : e] : r.next;
          if (!hn || kl.mesh(nk) != m) {  // last element (copy) of its mesh
            spans[(uint64_t)m * n_levels].elem_end = bu + ru;
            spans[(uint64_t)m * n_levels].group_end = bg + rg;
          }
          pk = key;
          hp = true;
        }
      }
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < tu; i += BLOCK) elem1[(uint64_t)bu + i] = s_key[i];
    __syncthreads();
    // elem2 / first_child2 staged by tile-local group index
    {
      uint32_t ru = (uint32_t)ex, rg = (uint32_t)(ex >> 32);
#pragma unroll
      for (int e = 0; e < EPT; ++e) {
        if ((uint32_t)e < r.cnt) {
          const uint32_t fl = (f >> (2 * e)) & 3u;
          if (fl & 1u) {
            if (fl & 2u) {
              s_key[rg] = kl.parent(r.kk[e]);
              s_val[rg] = bu + ru;
              ++rg;
            }
            ++ru;
          }
        }
      }
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < tg; i += BLOCK) {
      elem2[(uint64_t)bg + i] = s_key[i];
      first_child2[(uint64_t)bg + i] = s_val[i];
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------- level 1 from the bitmap
// The occupancy bitmap holds, per mesh, one bit per cell in Morton order, so
// its set bits in word order are the sorted unique keys and the nonzero bytes
// are the parent groups (the eight children of parent p are codes 8p..8p+7,
// one byte).  count -> scan of tile counts -> emit, each over tiles of 2048
// words.
constexpr int BM_WPT = 8;                 // words per thread (two 16-byte pieces)
constexpr int BM_TILE = BLOCK * BM_WPT;   // 2048 words
static_assert(BM_WPT % 4 == 0, "threads load whole 16-byte pieces");

__device__ inline uint32_t nonzero_bytes(uint32_t w) {
  const uint32_t t = (w & 0x7F7F7F7Fu) + 0x7F7F7F7Fu;  // bit 7 of a byte: low 7 bits nonzero
  return __popc((t | w) & 0x80808080u);
}

__device__ inline void load_words(const uint32_t* bits, uint64_t n_words, uint64_t w0,
                                  uint32_t (&w)[BM_WPT]) {
  if (w0 + BM_WPT <= n_words) {
#pragma unroll
    for (int q = 0; q < BM_WPT / 4; ++q) {
      const uint4 a = ((const uint4*)(bits + w0))[q];
      w[4 * q] = a.x; w[4 * q + 1] = a.y; w[4 * q + 2] = a.z; w[4 * q + 3] = a.w;
    }
  } else {
#pragma unroll
    for (int j = 0; j < BM_WPT; ++j) w[j] = w0 + j < n_words ? bits[w0 + j] : 0u;
  }
}

// A bitmap past the caches (one mesh's, LINES) is not read whole: the
// voxelization flags the 64-byte lines (512 cells) that it sets bits of, a byte
// a line, and the tiles are made of 128 flagged lines each, in order.  100,000
// triangles at 2048^3: 72 us in all and 22 more for the flags' stores, where
// counting and emitting over the 1.07 GB took 180 and 284 us.
constexpr int LINE_WORDS = BITMAP_LINE_BYTES / 4;
constexpr int TILE_LINES = BM_TILE / LINE_WORDS;
struct LineList {
  const uint32_t* line;  // flagged lines in order
  const uint32_t* n;     // their number
};
__device__ inline uint64_t line_tiles(const LineList& L) {
  return ((uint64_t)*L.n + TILE_LINES - 1) / TILE_LINES;
}
// The first bitmap word of this thread's eight in a tile (past n_words: none).
template <bool LINES>
__device__ inline uint64_t tile_words(const LineList& L, uint64_t tile, uint64_t n_words,
                                      uint32_t* s_line) {
  if (!LINES) return tile * BM_TILE + threadIdx.x * BM_WPT;
  static_assert(2 * BM_WPT == LINE_WORDS, "two threads a line");
  const uint64_t i = tile * TILE_LINES + (threadIdx.x >> 1);
  if (i >= *L.n) return n_words;
  const uint32_t line = L.line[i];
  if (s_line) s_line[threadIdx.x >> 1] = line;
  return (uint64_t)line * LINE_WORDS + (threadIdx.x & 1) * BM_WPT;
}

// Number of flagged lines per run of `per` pieces of LINE_PIECE flags.
constexpr int LINE_PIECE = BLOCK * 64;
constexpr uint32_t LINE_RUNS = 2048;
constexpr uint64_t LINE_GRID = 8192;
__device__ inline uint32_t load_flags(const uint8_t* flags, uint64_t n_lines, uint64_t i0,
                                      uint4 (&f)[4]) {
  uint32_t c = 0;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    f[q] = make_uint4(0u, 0u, 0u, 0u);
    if (i0 + 16 * q < n_lines) f[q] = ((const uint4*)(flags + i0))[q];  // (n_lines: whole tiles)
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) c += __popc(f[q].x) + __popc(f[q].y) + __popc(f[q].z) + __popc(f[q].w);
  return c;
}
__global__ __launch_bounds__(BLOCK) void k_line_count(const uint8_t* flags, uint64_t n_lines,
                                                      uint32_t per, uint32_t* run_count) {
  __shared__ uint32_t tmp[8];
  uint32_t c = 0;
  for (uint32_t k = 0; k < per; ++k) {
    uint4 f[4];
    c += load_flags(flags, n_lines, ((uint64_t)blockIdx.x * per + k) * LINE_PIECE + threadIdx.x * 64,
                    f);
  }
  uint32_t none = 0, t, u;
  block_excl_scan256_2(c, none, tmp, t, u);
  if (threadIdx.x == 0) run_count[blockIdx.x] = t;
}
__global__ __launch_bounds__(BLOCK) void k_line_list(const uint8_t* flags, uint64_t n_lines,
                                                     uint32_t per, const uint32_t* run_count,
                                                     uint32_t* line, uint32_t* n) {
  __shared__ uint32_t tmp[8];
  uint32_t before = 0, none = 0, t, u;
  for (uint32_t i = threadIdx.x; i < blockIdx.x; i += BLOCK) before += run_count[i];
  block_excl_scan256_2(before, none, tmp, t, u);
  uint64_t base = t;
  for (uint32_t k = 0; k < per; ++k) {
    const uint64_t i0 = ((uint64_t)blockIdx.x * per + k) * LINE_PIECE + threadIdx.x * 64;
    uint4 f[4];
    const uint32_t c = load_flags(flags, n_lines, i0, f);
    __syncthreads();  // tmp is read above
    uint32_t a = c, b = 0;
    block_excl_scan256_2(a, b, tmp, t, u);
    uint64_t o = base + a;
    if (c) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t w[4] = {f[q].x, f[q].y, f[q].z, f[q].w};
#pragma unroll
        for (int j = 0; j < 4; ++j)
          for (uint32_t r = w[j]; r; r &= r - 1u)
            line[o++] = (uint32_t)(i0 + 16 * q + 4 * j + (__builtin_ctz(r) >> 3));
      }
    }
    base += t;
  }
  if (blockIdx.x + 1 == gridDim.x && threadIdx.x == 0) *n = (uint32_t)base;
}

// Zeroes the 16-byte pieces of the words loaded by load_words that are not
// already zero.
__device__ inline void clear_words(uint32_t* bits, uint64_t n_words, uint64_t w0,
                                   const uint32_t (&w)[BM_WPT]) {
  if (w0 + BM_WPT <= n_words) {
#pragma unroll
    for (int q = 0; q < BM_WPT / 4; ++q)
      if (w[4 * q] | w[4 * q + 1] | w[4 * q + 2] | w[4 * q + 3])
        ((uint4*)(bits + w0))[q] = make_uint4(0u, 0u, 0u, 0u);
  } else {
#pragma unroll
    for (int j = 0; j < BM_WPT; ++j)
      if (w0 + j < n_words && w[j]) bits[w0 + j] = 0u;
  }
}

// Tile counts per thread in the scan: short chunks spread the loads over
// more workgroups (4 measured faster than 16, and 64, one workgroup for a
// res-1024 bitmap, slower still: its loads are latency-bound).
constexpr int SC_PER = 4;
constexpr int SC_CHUNK = BLOCK * SC_PER;     // 1024 tiles per scan workgroup

// Per tile: set bits, nonzero bytes, and the 4-byte units k_bm_emit will
// zero.
template <bool LINES>
__global__ __launch_bounds__(BLOCK) void k_bm_count(const uint32_t* bits, uint64_t n_words,
                                                    LineList L, uint32_t* tile_u, uint32_t* tile_g,
                                                    uint32_t* tile_r, uint64_t* scan_status,
                                                    uint32_t n_status) {
  __shared__ uint32_t tmp[8];
  // the tile-count scan's look-back words and ticket start at zero
  if (blockIdx.x == 0)
    for (uint32_t i = threadIdx.x; i < n_status; i += BLOCK) scan_status[i] = 0;
  const uint64_t tiles = LINES ? line_tiles(L) : gridDim.x;
  for (uint64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    const uint64_t w0 = tile_words<LINES>(L, tile, n_words, nullptr);
    uint32_t w[BM_WPT];
    load_words(bits, n_words, w0, w);
    // a: set bits (0-16) and the 4-byte units clear_words will zero (17-28);
    // b: nonzero bytes
    uint32_t a = 0, b = 0;
#pragma unroll
    for (int j = 0; j < BM_WPT; ++j) {
      a += __popc(w[j]);
      b += nonzero_bytes(w[j]);
    }
    if (w0 + BM_WPT <= n_words) {
#pragma unroll
      for (int q = 0; q < BM_WPT / 4; ++q)
        a += (w[4 * q] | w[4 * q + 1] | w[4 * q + 2] | w[4 * q + 3]) ? (4u << 17) : 0u;
    } else {
#pragma unroll
      for (int j = 0; j < BM_WPT; ++j) a += (uint32_t)(w[j] != 0) << 17;
    }
    uint32_t ta, tb;
    block_excl_scan256_2(a, b, tmp, ta, tb);  // only the totals are used
    if (threadIdx.x == 0) {
      tile_u[tile] = ta & 0x1FFFFu;
      tile_g[tile] = tb;
      tile_r[tile] = ta >> 17;
    }
    if (LINES) __syncthreads();
  }
}

// The counter slots' sums, by one wave.
__device__ inline void sum_counters(const unsigned long long* slots, unsigned long long* totals) {
  static_assert(COUNT_SLOTS == 64, "a lane per slot");
  const unsigned long long* slot = slots + threadIdx.x * COUNT_STRIDE;
  const uint64_t c = wave_sum((uint64_t)slot[COUNT_CELLS]);
  const uint64_t k = wave_sum((uint64_t)slot[COUNT_CHUNKS]);
  const uint64_t h = wave_sum((uint64_t)slot[COUNT_HITS]);
  if (threadIdx.x == 0) {
    totals[0] = c;
    totals[1] = k;
    totals[2] = h;
  }
}

// Exclusive scan of the tile counts in place, SC_CHUNK tiles per workgroup, chunk
// offsets by decoupled look-back (chunks claimed by ticket); totals to
// counts[0] (unique keys = level-1 elements) and counts[1] (groups = level-2
// elements); the bytes k_bm_emit will zero are added to *reset_bytes.
__global__ __launch_bounds__(BLOCK) void k_bm_scan(uint32_t* tile_u, uint32_t* tile_g,
                                                   const uint32_t* tile_r, uint32_t tiles,
                                                   LineList L, uint64_t* scan_status,
                                                   unsigned long long* counts,
                                                   unsigned long long* reset_bytes,
                                                   const unsigned long long* slots,
                                                   unsigned long long* totals) {
  __shared__ uint64_t tmp[4];
  __shared__ uint32_t s_chunk, s_base[2], s_reset[BLOCK / 64];
  if (blockIdx.x == 0 && threadIdx.x < 64) sum_counters(slots, totals);
  if (L.line) {  // flagged lines only: the later workgroups have no chunk
    tiles = (uint32_t)line_tiles(L);
    if ((uint64_t)blockIdx.x * SC_CHUNK >= tiles) return;
  }
  uint32_t* ticket = (uint32_t*)scan_status;  // word 0; chunk c uses words 2 + 2c, 3 + 2c
  if (threadIdx.x == 0) s_chunk = atomicAdd(ticket, 1u);
  __syncthreads();
  const uint32_t chunk = s_chunk;
  const uint32_t i0 = chunk * SC_CHUNK + threadIdx.x * SC_PER;
  uint32_t a[SC_PER], b[SC_PER];
#pragma unroll
  for (int j = 0; j < SC_PER; ++j) {
    const uint32_t i = i0 + j;
    const uint32_t c = i < tiles ? i : tiles - 1;
    a[j] = tile_u[c];
    b[j] = tile_g[c];
  }
  uint32_t su = 0, sg = 0, sr = 0;
#pragma unroll
  for (int j = 0; j < SC_PER; ++j)
    if (i0 + j < tiles) {
      su += a[j];
      sg += b[j];
      sr += tile_r[i0 + j];
    }
  for (int d = 32; d >= 1; d >>= 1) sr += __shfl_xor(sr, d);
  if (__lane_id() == 0) s_reset[threadIdx.x >> 6] = sr;
  uint64_t tot;
  const uint64_t ex = block_excl_scan256(((uint64_t)sg << 32) | su, tmp, tot);
  if (threadIdx.x < 2) {
    const uint32_t c = threadIdx.x == 0 ? (uint32_t)tot : (uint32_t)(tot >> 32);
    const uint32_t pre = lookback_exclusive(scan_status + 2 + threadIdx.x, 2, chunk, c, 1u);
    s_base[threadIdx.x] = pre;
    if ((uint64_t)(chunk + 1) * SC_CHUNK >= tiles) counts[threadIdx.x] = (unsigned long long)pre + c;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    uint64_t r = 0;
    for (int v = 0; v < BLOCK / 64; ++v) r += s_reset[v];
    if (r) atomicAdd(reset_bytes, (unsigned long long)(4 * r));
  }
  uint32_t ru = s_base[0] + (uint32_t)ex, rg = s_base[1] + (uint32_t)(ex >> 32);
#pragma unroll
  for (int j = 0; j < SC_PER; ++j) {
    const uint32_t i = i0 + j;
    if (i < tiles) {
      tile_u[i] = ru;
      tile_g[i] = rg;
      ru += a[j];
      rg += b[j];
    }
  }
}

__device__ inline uint32_t mesh_of_word(const uint64_t* bm_off, uint32_t n_meshes, uint64_t gw) {
  uint32_t lo = 0, hi = n_meshes;  // bm_off[lo] <= gw < bm_off[hi]
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (bm_off[mid] <= gw) lo = mid; else hi = mid;
  }
  return lo;
}

// One tile of 2048 words, which lies inside one mesh's bitmap region (the
// regions start on tile boundaries).  The tile's nonzero words are compacted
// into LDS in word order with the exclusive prefixes of their set bits (low
// 17 bits) and nonzero bytes (high 15 bits).  Then, 256 nonzero words per
// round, a lane takes one word and walks its set bits (unique keys, in order)
// and its nonzero bytes (groups) into LDS buffers, which the block writes out
// contiguously.  A lane per nonzero word keeps most lanes busy (a lane per
// bit would leave about four in five idle at surface densities), and staging
// turns the lanes' strided stores into whole cache lines.  A key is staged
// as its 16-bit bit index in the tile (the tile's first key is added at
// copy-out) and a group as its word in the round and byte in the word (its
// parent, first key and child mask are read back from the word), so the
// workgroup's LDS stays near 26 KB for either key width and six workgroups
// fit a CU.  A round with more than
// EMIT_CAP keys (dense tiles) stores its keys and groups directly.  The
// tile's words are zeroed after they are read.
constexpr uint32_t EMIT_CAP = 2048;
static_assert((EMIT_CAP & (EMIT_CAP - 1)) == 0, "the copy-out masks slot indices");
static_assert(BM_TILE % BLOCK == 0, "a round's words lie inside the tile's LDS arrays");
static_assert(BM_TILE == BITMAP_TILE_WORDS, "mesh regions start on tile boundaries");

struct BmSums {  // SUMS: what k_bm_scan does otherwise
  const uint32_t* tile_r;
  unsigned long long *counts, *reset_bytes, *totals;
  const unsigned long long* slots;
};
// SUMS: up to SUM_TILES tiles a workgroup adds up the tile counts before its
// own itself, 8 loads a thread, which saves the scan's launch (5 us).
constexpr uint64_t SUM_TILES = 2048;
template <typename K, bool LINES, bool SUMS>
__global__ __launch_bounds__(BLOCK) void k_bm_emit(uint32_t* bits, uint64_t n_words, LineList L,
                                                   BmSums sums, const uint64_t* bm_off, uint32_t n_meshes,
                                                   KeyLayout<K> kl, const uint32_t* tile_u,
                                                   const uint32_t* tile_g, K* elem1, K* elem2,
                                                   uint32_t* first_child2, uint8_t* kids2,
                                                   const unsigned long long* counts,
                                                   LevelSpan* spans, uint32_t n_levels,
                                                   MeshTreeState* state, uint64_t* status,
                                                   uint32_t* tickets) {
  __shared__ uint32_t tmp[8];
  __shared__ uint32_t s_word[BM_TILE], s_pre[BM_TILE];
  __shared__ uint16_t s_idx[BM_TILE], s_key[EMIT_CAP], s_grp[BLOCK * 4];
  __shared__ K s_kbase;  // key of the tile's bit 0
  __shared__ uint32_t s_line[LINES ? TILE_LINES : 1];
  const uint32_t l0 = threadIdx.x * BM_WPT;
  // the bitmap words and the tile's output offsets are loaded first, so that
  // the mesh lookup's dependent loads run while they are in flight
  uint32_t w[BM_WPT];
  uint64_t w0 = 0;
  if (!LINES) {
    w0 = tile_words<LINES>(L, blockIdx.x, n_words, s_line);
    load_words(bits, n_words, w0, w);
  }
  // SUMS: set bits and nonzero bytes before this tile, before the tile that
  // follows its mesh, and in all
  enum { BEFORE, MESH_END, ALL };
  __shared__ uint32_t s_sum[3][2][BLOCK / 64], s_reset[BLOCK / 64];
  uint32_t sum_u[3], sum_g[3], first_mesh = 0;
  uint64_t mesh_off = 0;
  if (SUMS) {
    const uint64_t tw0 = (uint64_t)blockIdx.x * BM_TILE;
    first_mesh = mesh_of_word(bm_off, n_meshes, tw0);
    mesh_off = bm_off[first_mesh];
    const uint64_t limit[3] = {blockIdx.x, bm_off[first_mesh + 1] / BM_TILE, gridDim.x};
    uint32_t u[SUM_TILES / BLOCK], g[SUM_TILES / BLOCK], r = 0;
#pragma unroll
    for (uint32_t j = 0; j < SUM_TILES / BLOCK; ++j) {
      const uint32_t i = j * BLOCK + threadIdx.x;
      u[j] = i < gridDim.x ? tile_u[i] : 0u;
      g[j] = i < gridDim.x ? tile_g[i] : 0u;
      if (blockIdx.x == 0 && i < gridDim.x) r += sums.tile_r[i];
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      uint32_t a = 0, b = 0;
#pragma unroll
      for (uint32_t j = 0; j < SUM_TILES / BLOCK; ++j) {
        const bool in = j * BLOCK + threadIdx.x < limit[k];
        a += in ? u[j] : 0u;
        b += in ? g[j] : 0u;
      }
      a = wave_sum_u32(a);
      b = wave_sum_u32(b);
      if (__lane_id() == 0) {
        s_sum[k][0][threadIdx.x >> 6] = a;
        s_sum[k][1][threadIdx.x >> 6] = b;
      }
    }
    if (blockIdx.x == 0) {
      r = wave_sum_u32(r);
      if (__lane_id() == 0) s_reset[threadIdx.x >> 6] = r;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      sum_u[k] = sum_g[k] = 0;
#pragma unroll
      for (int w = 0; w < BLOCK / 64; ++w) {
        sum_u[k] += s_sum[k][0][w];
        sum_g[k] += s_sum[k][1][w];
      }
    }
    if (blockIdx.x == 0 && threadIdx.x < 64) {
      sum_counters(sums.slots, sums.totals);
      if (threadIdx.x == 0) {
        sums.counts[0] = sum_u[ALL];
        sums.counts[1] = sum_g[ALL];
        uint64_t t = 0;
        for (int w = 0; w < BLOCK / 64; ++w) t += s_reset[w];
        *sums.reset_bytes += 4 * t;
      }
    }
  }
  const uint64_t n_unique = SUMS ? sum_u[ALL] : counts[0];
  {
    // the later levels' look-back words and tickets start at zero (as
    // k_level_clear leaves them), a slice per workgroup
    const uint64_t words = 2 * level_tiles(n_unique);
    const uint64_t per = (words + gridDim.x - 1) / gridDim.x;
    const uint64_t i1 = std::min<uint64_t>(words, (uint64_t)(blockIdx.x + 1) * per);
    for (uint64_t i = (uint64_t)blockIdx.x * per + threadIdx.x; i < i1; i += BLOCK) status[i] = 0;
    if (blockIdx.x == 0 && threadIdx.x < MAX_TICKETS) tickets[threadIdx.x] = 0;
  }
  if (LINES && blockIdx.x == 0 && threadIdx.x == 0) {
    // the one mesh's level-1 span, and its depth-1 root if that is one voxel
    spans[0].elem_first = spans[0].group_first = 0;
    spans[0].elem_end = (uint32_t)counts[0];
    spans[0].group_end = (uint32_t)counts[1];
    if (counts[0] == 1) {
      state[0].depth = 1;
      state[0].root_elem = 0;
    }
  }
  const uint64_t tiles = LINES ? line_tiles(L) : gridDim.x;
  for (uint64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    if (LINES) {
      w0 = tile_words<LINES>(L, tile, n_words, s_line);
      load_words(bits, n_words, w0, w);
    }
    const uint32_t bu = SUMS ? sum_u[BEFORE] : tile_u[tile],
                   bg = SUMS ? sum_g[BEFORE] : tile_g[tile];
    if (!LINES && threadIdx.x == 0) {
      const uint64_t tw0 = tile * BM_TILE;
      const uint32_t m = SUMS ? first_mesh : mesh_of_word(bm_off, n_meshes, tw0);
      const uint64_t off = SUMS ? mesh_off : bm_off[m];
      s_kbase = ((K)m << kl.cb) | ((K)(tw0 - off) << 5);
      if (tw0 == off) {
        // the mesh's first tile: its level-1 span ends where the next mesh's
        // first tile starts (every region is whole tiles) and, for a mesh whose
        // level 1 holds a single voxel, its depth-1 root (what
        // k_first_finalize does on the sort path)
        const uint64_t tn = bm_off[m + 1] / BM_TILE;
        const uint32_t ue = SUMS                ? sum_u[MESH_END]
                            : tn < gridDim.x ? tile_u[tn]
                                             : (uint32_t)counts[0];
        const uint32_t ge = SUMS                ? sum_g[MESH_END]
                            : tn < gridDim.x ? tile_g[tn]
                                             : (uint32_t)counts[1];
        LevelSpan& sp = spans[(uint64_t)m * n_levels];
        sp.elem_first = bu;
        sp.elem_end = ue;
        sp.group_first = bg;
        sp.group_end = ge;
        if (ue - bu == 1) {
          state[m].depth = 1;
          state[m].root_elem = bu;
        }
      }
    }
    clear_words(bits, n_words, w0, w);  // the bitmap is left clear for the next pass
    // a: set bits (0-16) and nonzero words (17-28); b: nonzero bytes
    uint32_t a = 0, b = 0;
#pragma unroll
    for (int j = 0; j < BM_WPT; ++j) {
      a += __popc(w[j]) + ((uint32_t)(w[j] != 0) << 17);
      b += nonzero_bytes(w[j]);
    }
    uint32_t ta, tb;
    block_excl_scan256_2(a, b, tmp, ta, tb);  // tmp is not used again
    {
      uint32_t pu = a & 0x1FFFFu, pg = b, pz = a >> 17;
#pragma unroll
      for (int j = 0; j < BM_WPT; ++j) {
        if (w[j]) {
          s_word[pz] = w[j];
          s_pre[pz] = pu | (pg << 17);  // pu <= 65535, pg <= 8191 for a nonzero word
          s_idx[pz] = (uint16_t)(l0 + j);
          ++pz;
        }
        pu += __popc(w[j]);
        pg += nonzero_bytes(w[j]);
      }
    }
    __syncthreads();
    const uint32_t nz = ta >> 17;
    const uint32_t pre_end = (ta & 0x1FFFFu) | (tb << 17);
    // key of a tile bit
    const K kbase = LINES ? (K)0 : s_kbase;
    auto key_of = [&](uint32_t b) -> K {
      return LINES ? ((K)s_line[b >> 9] << 9) | (K)(b & 511u) : kbase + (K)b;
    };
    for (uint32_t r0 = 0; r0 < nz; r0 += BLOCK) {
      const uint32_t r1 = r0 + BLOCK < nz ? r0 + BLOCK : nz;
      const uint32_t pre0 = s_pre[r0], pre1 = r1 < nz ? s_pre[r1] : pre_end;
      const uint32_t u0 = pre0 & 0x1FFFFu, nu = (pre1 & 0x1FFFFu) - u0;
      const uint32_t g0 = pre0 >> 17, ng = (pre1 >> 17) - g0;
      const bool stage = nu <= EMIT_CAP;  // the same for the whole block
      const uint32_t it = r0 + threadIdx.x;
      if (it < r1) {
        const uint32_t word = s_word[it], pre = s_pre[it];
        const uint32_t wb = (uint32_t)s_idx[it] << 5;  // tile bit index of the word's bit 0
        const uint32_t lu = (pre & 0x1FFFFu) - u0;
        // unique keys: the set bits in order
        if (stage) {
          uint32_t o = lu;
          for (uint32_t r = word; r; r &= r - 1u) s_key[o++] = (uint16_t)(wb | __builtin_ctz(r));
        } else {
          K* out = elem1 + (uint64_t)bu + u0 + lu;
          const K hi = key_of(wb);
          for (uint32_t r = word; r; r &= r - 1u) *out++ = hi | (K)__builtin_ctz(r);
        }
        // groups: the nonzero bytes in order, tested in turn (a loop over the
        // nonzero bytes runs as often as the wave's fullest word has them,
        // nearly always four).  A group's first child is the unique key of
        // the byte's lowest set bit (the set bits below it are those of the
        // lower bytes); its parent is parent(word's key 0) + byte index, its
        // child mask the byte itself.
        uint32_t lg = (pre >> 17) - g0;
        if (stage) {
#pragma unroll
          for (uint32_t b = 0; b < 4; ++b) {
            if ((word >> (8 * b)) & 0xFFu) s_grp[lg++] = (uint16_t)((threadIdx.x << 2) | b);
          }
        } else {
          const uint32_t pu_w = pre & 0x1FFFFu;
          const K phi = kl.parent(key_of(wb));
          const uint64_t d0 = (uint64_t)bg + g0;
#pragma unroll
          for (uint32_t b = 0; b < 4; ++b) {
            if ((word >> (8 * b)) & 0xFFu) {
              elem2[d0 + lg] = phi | (K)b;
              first_child2[d0 + lg] = bu + pu_w + (b ? __popc(word & ((1u << (8 * b)) - 1u)) : 0u);
              kids2[d0 + lg] = (uint8_t)(word >> (8 * b));
              ++lg;
            }
          }
        }
      }
      __syncthreads();
      // copy-out, four elements per thread per step: the LDS reads are issued
      // together (slots past the round's count read stale entries inside the
      // buffers and store nothing)
      if (stage) {
        K* dst = elem1 + (uint64_t)bu + u0;
        for (uint32_t i0 = threadIdx.x; i0 < nu; i0 += 4 * BLOCK) {
          uint32_t v[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) v[j] = s_key[(i0 + j * BLOCK) & (EMIT_CAP - 1)];
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (i0 + j * BLOCK < nu) dst[i0 + j * BLOCK] = key_of(v[j]);
        }
        // groups, ng <= 4 * BLOCK: one step
        const uint32_t i0 = threadIdx.x;
        uint32_t c[4], word[4], pre[4], idx[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) c[j] = s_grp[i0 + j * BLOCK] & (4 * BLOCK - 1);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uint32_t wi = r0 + (c[j] >> 2);  // r0 <= BM_TILE - BLOCK
          word[j] = s_word[wi];
          pre[j] = s_pre[wi];
          idx[j] = s_idx[wi];
        }
        const uint64_t d0 = (uint64_t)bg + g0;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (i0 + j * BLOCK < ng) {
            const uint32_t sh = 8 * (c[j] & 3u);
            const uint64_t d = d0 + i0 + j * BLOCK;
            elem2[d] = kl.parent(key_of((idx[j] << 5) | sh));
            first_child2[d] = bu + (pre[j] & 0x1FFFFu) + __popc(word[j] & ((1u << sh) - 1u));
            kids2[d] = (uint8_t)(word[j] >> sh);
          }
      }
      __syncthreads();
    }
  }
}

// Child masks of the level-2 elements from the unique keys of level 1 (the
// sort path; the bitmap path reads them off its bytes): one thread per group,
// whose members are at most eight consecutive keys.
template <typename K>
__global__ __launch_bounds__(BLOCK) void k_first_kids(const K* elem1, const K* elem2,
                                                      const uint32_t* first_child2,
                                                      const unsigned long long* counts,
                                                      KeyLayout<K> kl, uint8_t* kids2) {
  const uint64_t n1 = counts[0], n2 = counts[1], stride = (uint64_t)gridDim.x * BLOCK;
  for (uint64_t g = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; g < n2; g += stride) {
    const K P = elem2[g];
    const uint64_t f = first_child2[g];
    uint32_t mask = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const K e = f + j < n1 ? elem1[f + j] : (K)~(K)P;
      if (f + j < n1 && kl.parent(e) == P) mask |= 1u << (uint32_t)(e & 7);
    }
    kids2[g] = (uint8_t)mask;
  }
}

__global__ void k_first_finalize(const LevelSpan* spans, uint32_t n_meshes, uint32_t n_levels,
                                 MeshTreeState* state) {
  const uint32_t m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= n_meshes) return;
  const LevelSpan sp = spans[(uint64_t)m * n_levels];
  if (sp.elem_end - sp.elem_first == 1) {  // a single voxel: depth-1 tree
    state[m].depth = 1;
    state[m].root_elem = sp.elem_first;
  }
}

// ---------------------------------------------------------------- level l >= 2
// Level elements -> their group (group_l, NONE for roots and finished
// meshes), the next level's keys with their first child and child mask, the
// spans of this level, roots into state, and counts[level] (elements of the
// next level).
template <typename K>
struct LevelIo {
  int level;
  KeyLayout<K> kl;
  MeshTreeState* state;
  const K* elem;
  uint32_t* group;
  K* elem_next;
  uint32_t* first_child_next;
  uint8_t* kids_next;
  LevelSpan* spans;
  uint32_t n_levels;
};

// The keys before and after a tile, as far as its first and last threads
// look: a group has at most eight members.
constexpr int AHEAD = 8;
// The workgroup's barrier for what it shares in LDS alone: __syncthreads()
// also waits for the global stores in flight, which beside another stream's
// emission take 10 us and more (a tail of five levels 184 us in place of 18).
__device__ inline void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
template <typename K, int T, int E>
struct LevelLds {
  K key[T * E];  // the tile's keys, then its groups' keys
  K before, after[AHEAD];
  uint32_t val[T * E];
  uint8_t kid[T * E];
  uint32_t wave[T / 64];
  uint32_t base;
};

// One tile of up to T * E elements from element tb on, T threads; base_of
// (called by the first wave, all lanes) turns the tile's group count into its
// first group.  Returns the group count; S.key then holds the groups' keys.
// `resident`: S.key already holds the tile's keys, the whole level (the keys
// that a tile left there).  Ends behind a barrier.
template <typename K, int T, int E, typename F>
__device__ inline uint32_t level_tile(const LevelIo<K>& A, uint64_t n, uint64_t tb,
                                      LevelLds<K, T, E>& S, bool resident, F base_of) {
  const uint32_t tn = (uint32_t)(n - tb < T * E ? n - tb : T * E), l0 = threadIdx.x * E;
  const uint32_t cnt = l0 < tn ? (tn - l0 < E ? tn - l0 : E) : 0u;
  const uint64_t i0 = tb + l0;
  const KeyLayout<K> kl = A.kl;
  K kk[E];
  if (resident) {
#pragma unroll
    for (int e = 0; e < E; ++e) kk[e] = S.key[l0 + e];
  } else {
    load_consecutive(A.elem + (cnt ? i0 : 0), ((uintptr_t)A.elem & 15) == 0 && cnt, cnt, kk);
    if (threadIdx.x < AHEAD && tb + tn + threadIdx.x < n)
      S.after[threadIdx.x] = A.elem[tb + tn + threadIdx.x];
    if (threadIdx.x == T - 1 && tb > 0) S.before = A.elem[tb - 1];
#pragma unroll
    for (int e = 0; e < E; ++e) S.key[l0 + e] = kk[e];
    lds_barrier();
  }
  const bool has_prev = cnt && i0 > 0, has_next = cnt && i0 + cnt < n;
  // the key after the thread's run and beyond (inside the level)
  auto ahead = [&](uint32_t j) -> K {
    const uint32_t i = l0 + cnt + j;
    return i < tn ? S.key[i] : S.after[i - tn];
  };
  const K prev = !has_prev ? (K)0 : l0 > 0 ? S.key[l0 - 1] : S.before;
  const K next = !has_next ? (K)0 : ahead(0);
  // 4 flag bits per element: bit0 live (its mesh is still being built),
  // bit1 group head, bit2 root
  uint64_t f = 0;
  uint32_t ng = 0, mask_ahead = 0;
  {
    uint32_t last_m = 0xFFFFFFFFu, done = 0;
    K pk = prev;
    bool hp = has_prev;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      if ((uint32_t)e < cnt) {
        const K cur = kk[e];
        // only level 2 holds an element of a finished mesh: the group of a
        // single voxel (a later level's root is no group)
        if (A.level == 2) {
          const uint32_t m = kl.mesh(cur);
          if (m != last_m) {
            done = A.state[m].depth;
            last_m = m;
          }
        }
        if (done == 0) {
          const bool more = e + 1 < E && (uint32_t)(e + 1) < cnt;
          const uint32_t fl = level_flags_v(pk, cur, more ? kk[(e + 1) % E] : next, hp,
                                            more || has_next, kl) | 1u;
          f |= (uint64_t)fl << (4 * e);
          ng += (fl >> 1) & 1u;
        }
        pk = cur;
        hp = true;
      }
    }
    // the thread's last group may go on past its run: at most seven more keys
    if (ng) {
      const K P = kl.parent(pk);
      for (uint32_t j = 0; j < AHEAD - 1 && i0 + cnt + j < n; ++j) {
        const K key = ahead(j);
        if (kl.parent(key) != P) break;
        mask_ahead |= 1u << (uint32_t)(key & 7);
      }
    }
  }
  const uint32_t inc = wave_incl_scan_dpp(ng);
  if ((threadIdx.x & 63) == 63) S.wave[threadIdx.x >> 6] = inc;
  lds_barrier();
  uint32_t exg = inc - ng, tg = 0;
#pragma unroll
  for (uint32_t w = 0; w < T / 64; ++w) {
    const uint32_t x = S.wave[w];
    if (w < threadIdx.x >> 6) exg += x;
    tg += x;
  }
  if (threadIdx.x < 64) {
    const uint32_t b = base_of(tg);
    if (threadIdx.x == 0) S.base = b;
  }
  lds_barrier();
  const uint32_t bg = S.base;
  uint32_t gv[E];
  {
    uint32_t rg = exg;
    K pk = prev;
    bool hp = has_prev;
    uint32_t mask = 0;  // children of the thread's current group so far
#pragma unroll
    for (int e = 0; e < E; ++e) {
      gv[e] = NONE;
      if ((uint32_t)e < cnt) {
        const K key = kk[e];
        const uint64_t i = i0 + e;
        const uint32_t fl = (uint32_t)(f >> (4 * e)) & 15u;
        const uint32_t m = kl.mesh(key);
        LevelSpan& sp = A.spans[(uint64_t)m * A.n_levels + (uint32_t)(A.level - 1)];
        if (fl & 4u) {  // the only key of its mesh at this level: the root
          A.state[m].depth = (uint32_t)A.level;
          A.state[m].root_elem = (uint32_t)i;
          sp.elem_first = (uint32_t)i;
          sp.elem_end = (uint32_t)i + 1;
          sp.group_first = sp.group_end = 0;
        } else if (fl & 1u) {
          if (fl & 2u) {
            if (rg > exg) S.kid[rg - 1] = (uint8_t)mask;
            S.key[rg] = kl.parent(key);
            S.val[rg] = (uint32_t)i;
            ++rg;
            mask = 0;
          }
          mask |= 1u << (uint32_t)(key & 7);
          gv[e] = bg + rg - 1;
          const bool more = e + 1 < E && (uint32_t)(e + 1) < cnt;
          if (!hp || kl.mesh(pk) != m) {
            sp.elem_first = (uint32_t)i;
            sp.group_first = bg + rg - 1;
          }
          if (!(more || has_next) || kl.mesh(more ? kk[(e + 1) % E] : next) != m) {
            sp.elem_end = (uint32_t)i + 1;
            sp.group_end = bg + rg;
          }
        }
        pk = key;
        hp = true;
      }
    }
    if (rg > exg) S.kid[rg - 1] = (uint8_t)(mask | mask_ahead);
  }
  if (((uintptr_t)A.group & 15) == 0 && cnt == E) {
    uint4* q = (uint4*)(A.group + i0);
#pragma unroll
    for (int v = 0; v < E / 4; ++v)
      q[v] = make_uint4(gv[4 * v], gv[4 * v + 1], gv[4 * v + 2], gv[4 * v + 3]);
  } else {
#pragma unroll
    for (int e = 0; e < E; ++e)
      if ((uint32_t)e < cnt) A.group[i0 + e] = gv[e];
  }
  lds_barrier();
  for (uint32_t i = threadIdx.x; i < tg; i += T) {
    A.elem_next[(uint64_t)bg + i] = S.key[i];
    A.first_child_next[(uint64_t)bg + i] = S.val[i];
    A.kids_next[(uint64_t)bg + i] = S.kid[i];
  }
  lds_barrier();
  return tg;
}

// A level's tiles, claimed in order by ticket.  Workgroups past the tiles
// leave without a ticket and, when every tile has a workgroup, each takes one
// only: tickets on one address follow each other at about 6 ns, and a grid
// sized for the level's capacity holds mostly workgroups without a tile.
template <typename K, int E>
__device__ inline void level_pass(const LevelIo<K>& A, uint64_t n, LevelLds<K, BLOCK, E>& S,
                                  uint32_t* s_tile, uint64_t* status, uint32_t* ticket,
                                  uint32_t epoch, unsigned long long* count_next) {
  constexpr uint64_t T = BLOCK * E;
  const uint64_t tiles = (n + T - 1) / T;
  if (blockIdx.x >= tiles) return;
  const bool once = tiles <= gridDim.x;
  do {
    if (threadIdx.x == 0) *s_tile = atomicAdd(ticket, 1u);
    __syncthreads();
    const uint64_t tile = *s_tile;
    if (tile >= tiles) return;  // uniform over the workgroup
    level_tile<K, BLOCK, E>(A, n, tile * T, S, false, [&](uint32_t tg) {
      const uint32_t pre = lookback_exclusive_wave(status + 1, 2, tile, tg, epoch);
      if (threadIdx.x == 0 && tile + 1 == tiles) *count_next = (unsigned long long)pre + tg;
      return pre;
    });
  } while (!once);
}

template <typename K>
__global__ __launch_bounds__(BLOCK) void k_level_pass(LevelIo<K> A,
                                                      const unsigned long long* n_ptr,
                                                      uint64_t* status, uint32_t* ticket,
                                                      uint32_t epoch,
                                                      unsigned long long* count_next) {
  __shared__ union {
    LevelLds<K, BLOCK, EPT> big;
    LevelLds<K, BLOCK, EPT_SMALL> small;
  } S;
  __shared__ uint32_t s_tile;
  const uint64_t n = *n_ptr;
  if (n <= SMALL_ELEMS)
    level_pass<K, EPT_SMALL>(A, n, S.small, &s_tile, status, ticket, epoch, count_next);
  else
    level_pass<K, EPT>(A, n, S.big, &s_tile, status, ticket, epoch, count_next);
}

// Levels `first` .. n_levels in one workgroup, a tile per level: at these sizes
// (TAIL_TILE elements at most, by the grid) a launch and its look-back cost
// more than the work.  With several tiles in turn (levels to 32768 elements)
// it was slower than the launches: 63 us against 43 where the level is full.
constexpr int TAIL_THREADS = 1024, TAIL_EPT = 4, TAIL_TILE = TAIL_THREADS * TAIL_EPT;
template <typename K>
struct TailArgs {
  LevelIo<K> io;  // what the levels share
  int first, last;
  struct Level {
    K* elem;
    uint32_t* group;
    uint32_t* first_child;
    uint8_t* kids;
  } lv[24];  // level l at [l - 1], up to last + 1
};
template <typename K>
__global__ __launch_bounds__(TAIL_THREADS) void k_level_tail(TailArgs<K> A,
                                                             unsigned long long* counts) {
  __shared__ LevelLds<K, TAIL_THREADS, TAIL_EPT> S;
  uint64_t n = counts[A.first - 1];
  for (int l = A.first; l <= A.last && n; ++l) {
    LevelIo<K> io = A.io;
    io.level = l;
    io.elem = A.lv[l - 1].elem;
    io.group = A.lv[l - 1].group;
    io.elem_next = A.lv[l].elem;
    io.first_child_next = A.lv[l].first_child;
    io.kids_next = A.lv[l].kids;
    // a level leaves the next level's keys in LDS
    n = level_tile<K, TAIL_THREADS, TAIL_EPT>(io, n, 0, S, l > A.first,
                                              [](uint32_t) { return 0u; });
    if (threadIdx.x == 0) counts[l] = n;
  }
}

uint32_t grid_tiles(uint64_t cap, uint32_t blocks) {
  const uint64_t tiles = (cap + TILE - 1) / TILE;
  return (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(tiles, blocks));
}

}  // namespace

size_t level_tmp_bytes(uint64_t cap) {
  return 256 + 2 * level_tiles(std::max<uint64_t>(cap, 1)) * sizeof(uint64_t);
}

template <typename K>
void launch_level_first(const K* sorted, const unsigned long long* n_sorted, uint64_t cap,
                        KeyLayout<K> kl, LevelArrays l1, LevelArrays l2,
                        unsigned long long* counts, LevelSpan* spans1, uint32_t n_levels,
                        uint32_t blocks, void* tmp, hipStream_t s) {
  uint32_t* tickets = (uint32_t*)tmp;
  uint64_t* status = (uint64_t*)((char*)tmp + 256);
  const uint64_t tiles = level_tiles(std::max<uint64_t>(cap, 1));
  const uint32_t cg = (uint32_t)std::min<uint64_t>(2048, (2 * tiles + BLOCK - 1) / BLOCK);
  hipLaunchKernelGGL(k_level_clear, dim3(std::max<uint32_t>(cg, 1)), dim3(BLOCK), 0, s, status,
                     tickets, n_sorted);
  hipLaunchKernelGGL(k_first_pass<K>, dim3(grid_tiles(cap, blocks)), dim3(BLOCK), 0, s, sorted,
                     n_sorted, kl, (K*)l1.elem, (K*)l2.elem, l2.first_child,
                     spans1, n_levels, status, tickets, 1u, counts);
  if (l2.kids) {
    const uint64_t kb = std::min<uint64_t>((cap + BLOCK - 1) / BLOCK, 8192);
    hipLaunchKernelGGL(k_first_kids<K>, dim3((uint32_t)std::max<uint64_t>(1, kb)), dim3(BLOCK), 0,
                       s, (const K*)l1.elem, (const K*)l2.elem,
                       (const uint32_t*)l2.first_child, (const unsigned long long*)counts, kl,
                       l2.kids);
  }
}

size_t bitmap_level_tmp_bytes(uint64_t n_words) {
  const uint64_t tiles = (std::max<uint64_t>(n_words, 1) + BM_TILE - 1) / BM_TILE;
  const uint64_t chunks = (tiles + SC_CHUNK - 1) / SC_CHUNK;
  return 3 * tiles * sizeof(uint32_t) + 256 + (2 + 2 * chunks) * sizeof(uint64_t) + 64;
}

template <typename K>
void launch_level_first_bitmap(uint32_t* bits, uint64_t n_words, const uint64_t* bm_off,
                               uint32_t n_meshes, KeyLayout<K> kl, LevelArrays l1,
                               LevelArrays l2, unsigned long long* counts, LevelSpan* spans1,
                               uint32_t n_levels, MeshTreeState* state, void* tmp,
                               void* lvl_tmp, unsigned long long* reset_bytes,
                               const unsigned long long* slots, unsigned long long* totals,
                               const uint8_t* line_flags, uint32_t* line_list, hipStream_t s) {
  const uint64_t tiles = (std::max<uint64_t>(n_words, 1) + BM_TILE - 1) / BM_TILE;
  const uint64_t chunks = (tiles + SC_CHUNK - 1) / SC_CHUNK;
  uint32_t* tile_u = (uint32_t*)tmp;
  uint32_t* tile_g = tile_u + tiles;
  uint32_t* tile_r = tile_g + tiles;
  uint64_t* scan_status =
      (uint64_t*)((char*)tmp + ((3 * tiles * sizeof(uint32_t) + 255) / 256) * 256);
  const uint32_t n_status = (uint32_t)(2 + 2 * chunks);
  uint32_t* tickets = (uint32_t*)lvl_tmp;
  uint64_t* status = (uint64_t*)((char*)lvl_tmp + 256);
  auto run = [&](auto lines, auto sums, const LineList& L, uint32_t grid) {
    constexpr bool LINES = decltype(lines)::value, SUMS = decltype(sums)::value;
    hipLaunchKernelGGL(k_bm_count<LINES>, dim3(grid), dim3(BLOCK), 0, s, bits, n_words, L, tile_u,
                       tile_g, tile_r, scan_status, n_status);
    if (!SUMS)
      hipLaunchKernelGGL(k_bm_scan, dim3((uint32_t)chunks), dim3(BLOCK), 0, s, tile_u, tile_g,
                       (const uint32_t*)tile_r, (uint32_t)tiles, L, scan_status, counts,
                       reset_bytes, slots, totals);
    // the emission also writes the level-1 spans and depth-1 roots, and clears
    // the later levels' look-back words and tickets (launch_levels)
    const BmSums bs{tile_r, counts, reset_bytes, totals, slots};
    hipLaunchKernelGGL((k_bm_emit<K, LINES, SUMS>), dim3(grid), dim3(BLOCK), 0, s, bits, n_words,
                       L, bs, bm_off, n_meshes, kl, (const uint32_t*)tile_u, (const uint32_t*)tile_g,
                       (K*)l1.elem, (K*)l2.elem, l2.first_child, l2.kids,
                       (const unsigned long long*)counts, spans1, n_levels, state, status,
                       tickets);
  };
  if (!line_flags) {
    if (tiles <= SUM_TILES) run(std::false_type{}, std::true_type{}, LineList{}, (uint32_t)tiles);
    else run(std::false_type{}, std::false_type{}, LineList{}, (uint32_t)tiles);
    return;
  }
  // runs of flags: at least a piece each (tile_g holds their counts for now)
  const uint64_t n_lines = n_words / LINE_WORDS, pieces = (n_lines + LINE_PIECE - 1) / LINE_PIECE;
  const uint32_t per = (uint32_t)((pieces + LINE_RUNS - 1) / LINE_RUNS);
  const uint32_t runs = (uint32_t)((pieces + per - 1) / per);
  uint32_t* n = (uint32_t*)(scan_status + n_status);
  hipLaunchKernelGGL(k_line_count, dim3(runs), dim3(BLOCK), 0, s, line_flags, n_lines, per, tile_g);
  hipLaunchKernelGGL(k_line_list, dim3(runs), dim3(BLOCK), 0, s, line_flags, n_lines, per,
                     (const uint32_t*)tile_g, line_list, n);
  run(std::true_type{}, std::false_type{}, LineList{line_list, n},
      (uint32_t)std::min<uint64_t>(tiles, LINE_GRID));
}

void launch_level_first_finalize(const LevelSpan* spans, uint32_t n_meshes, uint32_t n_levels,
                                 MeshTreeState* state, hipStream_t s) {
  hipLaunchKernelGGL(k_first_finalize, dim3((n_meshes + 63) / 64), dim3(64), 0, s, spans,
                     n_meshes, n_levels, state);
}

template <typename K>
void launch_levels(KeyLayout<K> kl, const LevelArrays* lv, uint32_t n_levels,
                   unsigned long long* counts, LevelSpan* spans, MeshTreeState* state,
                   uint32_t blocks, void* tmp, hipStream_t s) {
  uint32_t* tickets = (uint32_t*)tmp;
  uint64_t* status = (uint64_t*)((char*)tmp + 256);
  LevelIo<K> io{2, kl, state, nullptr, nullptr, nullptr, nullptr, nullptr, spans, n_levels};
  uint32_t l = 2;
  for (; l <= n_levels && lv[l].cap > TAIL_TILE; ++l) {
    io.level = (int)l;
    io.elem = (const K*)lv[l].elem;
    io.group = lv[l].elem_group;
    io.elem_next = (K*)lv[l + 1].elem;
    io.first_child_next = lv[l + 1].first_child;
    io.kids_next = lv[l + 1].kids;
    // counts[l - 1] = elements of this level; counts[l] = elements of the next
    const uint32_t grid =
        (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(level_tiles(lv[l].cap), blocks));
    hipLaunchKernelGGL(k_level_pass<K>, dim3(grid), dim3(BLOCK), 0, s, io,
                       (const unsigned long long*)counts + (l - 1), status, tickets + (l - 1), l,
                       counts + l);
  }
  if (l > n_levels) return;
  TailArgs<K> t{};
  t.io = io;
  t.first = (int)l;
  t.last = (int)n_levels;
  for (uint32_t k = l; k <= n_levels + 1; ++k)
    t.lv[k - 1] = {(K*)lv[k].elem, lv[k].elem_group, lv[k].first_child, lv[k].kids};
  hipLaunchKernelGGL(k_level_tail<K>, dim3(1), dim3(TAIL_THREADS), 0, s, t, counts);
}

template void launch_level_first<uint32_t>(const uint32_t*, const unsigned long long*, uint64_t,
                                           KeyLayout<uint32_t>, LevelArrays, LevelArrays,
                                           unsigned long long*, LevelSpan*, uint32_t, uint32_t,
                                           void*, hipStream_t);
template void launch_level_first<uint64_t>(const uint64_t*, const unsigned long long*, uint64_t,
                                           KeyLayout<uint64_t>, LevelArrays, LevelArrays,
                                           unsigned long long*, LevelSpan*, uint32_t, uint32_t,
                                           void*, hipStream_t);
template void launch_level_first_bitmap<uint32_t>(uint32_t*, uint64_t, const uint64_t*,
                                                  uint32_t, KeyLayout<uint32_t>, LevelArrays,
                                                  LevelArrays, unsigned long long*, LevelSpan*,
                                                  uint32_t, MeshTreeState*, void*, void*,
                                                  unsigned long long*, const unsigned long long*,
                                                  unsigned long long*, const uint8_t*, uint32_t*,
                                                  hipStream_t);
template void launch_level_first_bitmap<uint64_t>(uint32_t*, uint64_t, const uint64_t*,
                                                  uint32_t, KeyLayout<uint64_t>, LevelArrays,
                                                  LevelArrays, unsigned long long*, LevelSpan*,
                                                  uint32_t, MeshTreeState*, void*, void*,
                                                  unsigned long long*, const unsigned long long*,
                                                  unsigned long long*, const uint8_t*, uint32_t*,
                                                  hipStream_t);
template void launch_levels<uint32_t>(KeyLayout<uint32_t>, const LevelArrays*, uint32_t,
                                      unsigned long long*, LevelSpan*, MeshTreeState*, uint32_t,
                                      void*, hipStream_t);
template void launch_levels<uint64_t>(KeyLayout<uint64_t>, const LevelArrays*, uint32_t,
                                      unsigned long long*, LevelSpan*, MeshTreeState*, uint32_t,
                                      void*, hipStream_t);

}  // namespace svo
