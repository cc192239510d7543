// k_attrs.hip -- node records, neighbors and vertex / edge / face records.
//
// Node records (createNode_1 / createNode_2 / createRemainNode,
// SVO.cu:237-339) are written after the level phase has fixed every node
// count, in output order, from the level arrays:
//   code    = (group parent << 3) | k
//   origin  = gridOrigin + width * (float)decode(code)   per axis
//   isLeaf  = false only for occupied nodes above level 1
//   childs  = child level offset + 8 * (rank of the node's code in its level) + c
//   parent  = the parent group's node in the level above
// The root is its level's single code.  Node arrays are
// structure-of-arrays; the reference's 168-byte records are produced on copy.
//
// Neighbors (SVO.cu:522-565).  REFERENCE: the stored table holds UINT_MAX
// except root[13] = root (findNeighbors<false> writes a local copy,
// SVO.cu:535-542).  INTENDED: top-down, nb[s] = childs of the parent-level
// neighbor given by the neighbor LUTs (closed form of MortonLUT.h:531-597).
//
// Vertex / edge records (determineNodeVertex / determineNodeEdge +
// thrust::unique, SVO.cu:586-728).  REFERENCE: 8 corners w*(i&1, i>>1&1,
// i>>2&1) and 12 absolute edges per node, owner = the last stored neighbor of
// the sharing cells (600-603, 669-672), which is the node itself because the
// stored table has no other entries (root[13] is the root); a record equal to
// its predecessor is dropped (uniqueVert / uniqueEdge).  INTENDED: a vertex,
// edge or face is kept by the same-level sharing node with the smallest
// index.  A word per node says which it keeps; count -> scan -> write,
// node-major.
#include <algorithm>
#include <type_traits>

#include "svo_internal.h"
#include "svo_scan.h"

namespace svo {
namespace {

constexpr int BLOCK = 256;

// Grid-stride (n may exceed what one launch can index: 108 bytes of
// neighbors per node are 2^32 words at 160M nodes).  p is 16-byte aligned.
__global__ void k_fill_u32(uint32_t* p, uint32_t v, uint64_t n) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x * 4;
  for (uint64_t i = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4; i < n; i += stride) {
    if (i + 3 < n) {
      store_stream(reinterpret_cast<uint4*>(p + i), make_uint4(v, v, v, v));
    } else {
      for (uint64_t j = i; j < n; ++j) p[j] = v;
    }
  }
}

// ---------------------------------------------------------------- vertex / edge / face
// Edge endpoints in units of the node width, in the order of SVO.cu:638-663.
#define SVO_EDGE_ENDS                                                                           \
  {{{0, 0, 0}, {0, 1, 0}}, {{0, 1, 0}, {1, 1, 0}}, {{1, 1, 0}, {1, 0, 0}},                      \
   {{1, 0, 0}, {0, 0, 0}}, {{0, 0, 1}, {0, 1, 1}}, {{0, 1, 1}, {1, 1, 1}},                      \
   {{1, 1, 1}, {1, 0, 1}}, {{1, 0, 1}, {0, 0, 1}}, {{0, 0, 0}, {0, 0, 1}},                      \
   {{0, 1, 0}, {0, 1, 1}}, {{1, 1, 0}, {1, 1, 1}}, {{1, 0, 0}, {1, 0, 1}}}
constexpr uint8_t EDGE_ENDS[12][2][3] = SVO_EDGE_ENDS;  // for tables built when compiling
__constant__ uint8_t EDGE_OFS[12][2][3] = SVO_EDGE_ENDS;
#undef SVO_EDGE_ENDS
// Faces: -x, +x, -y, +y, -z, +z as (lo corner, hi corner) and the cell across.
constexpr uint8_t FACE_ENDS[6][2][3] = {{{0, 0, 0}, {0, 1, 1}}, {{1, 0, 0}, {1, 1, 1}},
                                        {{0, 0, 0}, {1, 0, 1}}, {{0, 1, 0}, {1, 1, 1}},
                                        {{0, 0, 0}, {1, 1, 0}}, {{0, 0, 1}, {1, 1, 1}}};
constexpr int FACE_SLOT[6] = {12, 14, 10, 16, 4, 22};

// origin + Vector3f(0|w, 0|w, 0|w), with the bare origin for the zero offset
// (SVO.cu:640-662).
__device__ inline void offset_point(const float* o, float w, const uint8_t* ofs, float* p) {
  const bool bare = !ofs[0] && !ofs[1] && !ofs[2];
#pragma unroll
  for (int a = 0; a < 3; ++a) p[a] = bare ? o[a] : o[a] + (ofs[a] ? w : 0.0f);
}

__device__ inline bool eq3(const float* a, const float* b) {
  return a[0] == b[0] && a[1] == b[1] && a[2] == b[2];
}

struct NodeGeom {
  float o[3];
  float w;
};
__device__ inline NodeGeom load_geom(const NodeArrays& n, uint64_t t) {
  NodeGeom g;
  g.o[0] = n.origin[3 * t];
  g.o[1] = n.origin[3 * t + 1];
  g.o[2] = n.origin[3 * t + 2];
  g.w = n.width[t];
  return g;
}

__device__ inline void ref_corner(float w, int j, float* p) {
  p[0] = w * (float)(j & 1);
  p[1] = w * (float)((j >> 1) & 1);
  p[2] = w * (float)((j >> 2) & 1);
}
__device__ inline void ref_edge(const NodeGeom& g, int i, float* a, float* b) {
  offset_point(g.o, g.w, EDGE_OFS[i][0], a);
  offset_point(g.o, g.w, EDGE_OFS[i][1], b);
}
__device__ inline bool edge_eq(const float* a0, const float* b0, const float* a1, const float* b1) {
  return (eq3(a0, a1) && eq3(b0, b1)) || (eq3(a0, b1) && eq3(b0, a1));
}

constexpr uint32_t LINE = 32;  // words of a cache line

// Writes words [w0, w0 + n) of dst, value(i) the word w0 + i: 16-byte pieces,
// single words where a piece lies across either end; four(i) gives the words
// i .. i + 3 at once.  dst is 16-byte aligned.  `stream`: past the caches.
template <typename F, typename F4>
__device__ inline void write_words(uint32_t* dst, uint64_t w0, uint32_t n, uint32_t tid,
                                   uint32_t threads, F value, F4 four, bool stream = true) {
  // from the cache line that w0 lies in: a wave's 1024 bytes are whole lines
  const uint32_t head = (uint32_t)w0 & (LINE - 1);
  uint32_t* p = dst + (w0 - head);
  for (uint32_t q = tid; 4 * q < head + n; q += threads) {
    const uint32_t i = 4 * q - head;  // wraps for words before w0
    if (4 * q + 3 < head) continue;
    if (4 * q >= head && i + 4 <= n) {
      if (stream) store_stream((uint4*)p + q, four(i));
      else ((uint4*)p)[q] = four(i);
    } else {
      for (uint32_t j = 0; j < 4; ++j)
        if (i + j < n) p[4 * (uint64_t)q + j] = value(i + j);
    }
  }
}
template <typename F>
__device__ inline void write_words(uint32_t* dst, uint64_t w0, uint32_t n, uint32_t tid,
                                   uint32_t threads, F value, bool stream = true) {
  write_words(
      dst, w0, n, tid, threads, value,
      [&](uint32_t i) {
        return make_uint4(value(i), value(i + 1), value(i + 2), value(i + 3));
      },
      stream);
}

// ---------------------------------------------------------------- emission
// Everything a pass outputs, in one launch.  The outputs are bound by their
// stores (169 bytes a node and 464 of reference records against about 2 read),
// and what the memory reaches depends on
//  * how close together the stores in flight lie: one 16-byte store per thread
//    with workgroups in address order runs at the rate of a plain fill
//    (6.7 TB/s), 4 / 8 stores per thread reach 5.9 / 5.6, a grid-stride loop
//    4.7;
//  * what a store waits for: origins and widths (16 bytes a node) read back
//    from memory that the writes keep busy held the edge records at 3.8 TB/s.
// So the arrays are written by consecutive workgroups in output order: the
// node arrays of rows of ROW nodes (a thread computes a node into LDS, then
// the workgroup writes 16-byte pieces), then edge records (two pieces a
// thread), vertex records, neighbor slots and voxel codes (one piece a
// thread).  Each part recomputes what it needs of its nodes from the level
// arrays, a few bytes per group of eight nodes that the caches hold.
// Measured on 16.1 M nodes with records (10.2 GB): 1,510 us, 6.7 TB/s; a node
// kernel per level beside a fill, then records from origins and widths, took
// 2,070 us.
constexpr int ROW = 512;  // nodes per row = threads per workgroup
constexpr int EDGE_BLOCKS = 21;  // workgroups per 2 * ROW nodes
constexpr int VERT_BLOCKS = 8;   // workgroups per row
constexpr uint32_t BLOCKS_PER_LAUNCH = 1u << 22;  // below 2^32 threads per launch
constexpr int REC_NODES = 2 * ROW / 21 + 2;  // nodes that a workgroup's edge pieces touch
constexpr int REC_VALS = 12;  // words per node in LDS: origin (bare, + 0, + w) x 3, owner, padding

// Read-only data through the scalar cache: uniform addresses become scalar loads.
template <typename T>
__device__ inline const __attribute__((address_space(4))) T* scalar_ptr(const T* p) {
  return (const __attribute__((address_space(4))) T*)p;
}

// Index of the segment that holds node t (the same t in every lane): the wave
// compares 64 segment starts at a time.
__device__ inline uint32_t find_seg(const uint32_t* seg_first, uint32_t n_segs, uint32_t t) {
  uint32_t lo = 0, n = n_segs;
  const uint32_t lane = __lane_id();
  while (true) {
    const uint32_t step = (n + 63) / 64, i = lane * step;
    const bool at = i < n && seg_first[lo + i] <= t;
    const uint32_t last = 63u - (uint32_t)__builtin_clzll(__ballot(at));  // seg_first[lo] <= t
    lo += last * step;
    if (step == 1) return __builtin_amdgcn_readfirstlane(lo);
    n = n - last * step < step ? n - last * step : step;
  }
}

// Runs body(seg, d) for the lanes' nodes t (in ascending lane order; at least
// t_first), d the node's place in its segment, one segment at a time with the
// segment uniform over the wave.
template <typename F>
__device__ inline void for_segments(const NodeSeg* segs, const uint32_t* seg_first,
                                    uint32_t n_segs, uint32_t t_first, uint32_t t, bool active,
                                    F body) {
  const auto* sg = scalar_ptr(segs) + find_seg(seg_first, n_segs, t_first);
  while (__any(active)) {
    if (active && t < sg->t1) {
      body(sg, t - sg->t0);
      active = false;
    }
    ++sg;
  }
}

template <typename K>
__device__ inline uint32_t axis_of(K code, uint32_t a) {
  return sizeof(K) == 4 ? compact3_32((uint32_t)code >> a)
                        : (uint32_t)compact3_64((uint64_t)code >> a);
}

// Edge piece p (words 4p .. 4p + 3 of a node's 84): the four words' LDS slots,
// four bits each.  Slot a is the bare origin of axis a (the zero offset,
// SVO.cu:640-662), 3 + a origin + 0, 6 + a origin + width, 9 the owner.
struct PieceTable {
  uint16_t slots[21];
};
constexpr PieceTable make_piece_table() {
  PieceTable t{};
  for (int p = 0; p < 21; ++p) {
    uint32_t v = 0;
    for (int k = 0; k < 4; ++k) {
      const int word = 4 * p + k, edge = word / 7, c = word % 7;
      uint32_t slot = 9;
      if (c < 6) {
        const uint8_t(&e)[3] = EDGE_ENDS[edge][c / 3];
        const int a = c % 3;
        slot = !e[0] && !e[1] && !e[2] ? a : e[a] ? 6 + a : 3 + a;
      }
      v |= slot << (4 * k);
    }
    t.slots[p] = (uint16_t)v;
  }
  return t;
}
__constant__ PieceTable PIECES = make_piece_table();

// LDS values of one axis of a node's records
__device__ inline void stage_axis(uint32_t* v, uint32_t a, float o, float w) {
  v[a] = __float_as_uint(o);
  v[3 + a] = __float_as_uint(o + 0.0f);
  v[6 + a] = __float_as_uint(o + w);
}

// Piece p of a row's edge records from the staged values of its nodes, the
// first of them node `f` of the row; s_piece holds PIECES.
__device__ inline uint4 edge_piece(const uint32_t* s_val, const uint32_t* s_piece, uint32_t f,
                                   uint32_t p) {
  const uint32_t n = p / 21, slots = s_piece[p - 21 * n];
  const uint32_t* v = s_val + REC_VALS * (n - f);
  return make_uint4(v[slots & 15], v[(slots >> 4) & 15], v[(slots >> 8) & 15], v[slots >> 12]);
}

__device__ inline uint4 vert_piece(float w, uint32_t j, uint32_t owner) {
  float p[3];
  ref_corner(w, (int)j, p);
  return make_uint4(__float_as_uint(p[0]), __float_as_uint(p[1]), __float_as_uint(p[2]), owner);
}

// Node arrays of one row.
template <typename K>
__device__ inline void emit_nodes(const EmitArgs<K>& A, uint64_t row, uint32_t* lds) {
  // LDS: children base, parent, width, origin, code (two words), leaf bytes
  uint32_t *s_ch = lds, *s_par = lds + ROW, *s_w = lds + 2 * ROW, *s_org = lds + 3 * ROW,
           *s_code = lds + 6 * ROW;
  uint8_t* s_leaf = (uint8_t*)(lds + 8 * ROW);
  const uint64_t t0 = row * ROW;
  const uint32_t i = threadIdx.x, t = (uint32_t)t0 + i;
  const bool wide = A.out.code_bytes == 8;
  for_segments(A.segs, A.seg_first, A.n_segs, t & ~63u, t, t < A.n_nodes,
               [&](auto* sg, uint32_t d) {
    const uint32_t kind = sg->level_kind, level = kind & 255u;
    const float w = sg->width;
    uint32_t parent = NONE, child = NONE;
    bool leaf = level == 1;
    const K* elem = (const K*)sg->elem;
    K code;
    if (kind & SEG_ROOT) {
      code = A.kl.code(elem[0]);
      if (level >= 2) child = sg->child0;
    } else {
      const uint32_t g = d >> 3, k = d & 7;
      const K P = elem[g];
      const uint32_t fc = sg->first_child[g], kids = sg->kids[g];
      parent = sg->parent0;
      if (!(kind & SEG_ROOT_CHILD)) parent += 8 * sg->group[g] + (uint32_t)(P & 7);
      code = (A.kl.code(P) << 3) | (K)k;
      const bool real = (kids >> k) & 1u;
      leaf = leaf || !real;
      if (real && level >= 2) child = sg->child0 + 8 * (fc + __popc(kids & ((1u << k) - 1u)));
    }
    s_ch[i] = child;
    s_par[i] = parent;
    s_w[i] = __float_as_uint(w);
    // gridOrigin + width * Vector3f(x, y, z), per axis (SVO.cu:262)
#pragma unroll
    for (uint32_t a = 0; a < 3; ++a)
      s_org[3 * i + a] = __float_as_uint(sg->origin[a] + w * (float)axis_of(code, a));
    if (wide) {
      s_code[2 * i] = (uint32_t)code;
      s_code[2 * i + 1] = (uint32_t)((uint64_t)code >> 32);
    } else {
      s_code[i] = (uint32_t)code;
    }
    s_leaf[i] = leaf ? 1 : 0;
  });
  __syncthreads();
  const uint64_t n = A.n_nodes - t0 < ROW ? A.n_nodes - t0 : ROW;  // nodes of the row
  // children: two pieces per node
#pragma unroll
  for (uint32_t u = 0; u < 2; ++u) {
    const uint32_t q = u * ROW + i, ln = q >> 1;
    if (ln < n) {
      const uint32_t b = s_ch[ln], c = b + 4 * (q & 1);
      store_stream((uint4*)(A.out.childs + 8 * t0) + q,
                   b == NONE ? make_uint4(NONE, NONE, NONE, NONE)
                             : make_uint4(c, c + 1, c + 2, c + 3));
    }
  }
  // the other arrays: pieces of ROW / 4 words each (origin 3, parent, width,
  // code 1 or 2), then the leaf bytes
  auto put = [&](const uint32_t* src, void* dst, uint32_t words, uint32_t q) {
    if (4 * q < n * words)
      store_stream((uint4*)((uint32_t*)dst + words * t0) + q, ((const uint4*)src)[q]);
  };
  constexpr uint32_t Q = ROW / 4;
  if (i < 3 * Q) put(s_org, A.out.origin, 3, i);
  else put(s_par, A.out.parent, 1, i - 3 * Q);
  if (i < Q) put(s_w, A.out.width, 1, i);
  else if (i < 3 * Q) {
    if (wide) put(s_code, A.out.code, 2, i - Q);
    else if (i < 2 * Q) put(s_code, A.out.code, 1, i - Q);
  } else if (16 * (i - 3 * Q) < n && i < 3 * Q + ROW / 16) {
    store_stream((uint4*)(A.out.is_leaf + t0) + (i - 3 * Q), ((const uint4*)s_leaf)[i - 3 * Q]);
  }
}

// Piece q of the neighbor slots, the reference's: NONE but for the root's own
// slot 13 (findNeighbors<true>, SVO.cu:528-529).  The root of a pass of one
// mesh is its last node; with more roots k_root_slots writes their slots
// afterwards, so that no fill waits for a lookup.
template <typename K>
__device__ inline void emit_neighbors(const EmitArgs<K>& A, uint64_t q) {
  if (4 * q >= 27 * A.n_nodes) return;
  uint4 v = make_uint4(NONE, NONE, NONE, NONE);
  if (A.n_roots == 1 && A.n_nodes > 1) {
    const uint32_t root = (uint32_t)A.n_nodes - 1;
    const uint64_t c = 27 * (A.n_nodes - 1) + 13 - 4 * q;  // wraps far up past the slot
    if (c == 0) v.x = root;
    else if (c == 1) v.y = root;
    else if (c == 2) v.z = root;
    else if (c == 3) v.w = root;
  }
  store_stream((uint4*)A.out.neighbors + q, v);
}

__global__ void k_root_slots(const NodeSeg* segs, uint32_t n_segs, NodeArrays out) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n_segs || (out.skip && *out.skip)) return;
  const uint32_t kind = segs[s].level_kind;
  if ((kind & SEG_ROOT) && (kind & 255u) >= 2)
    out.neighbors[27 * (uint64_t)segs[s].t0 + 13] = segs[s].local0;
}

// The workgroup stages the 10 values that a node's edge words are made of
// (three per axis and the owner) and builds its pieces from them: 21 of them
// per node, EDGE_BLOCKS workgroups of two pieces a thread per 2 * ROW nodes.
template <typename K>
__device__ inline void emit_edges(const EmitArgs<K>& A, uint32_t row, uint32_t block,
                                  uint32_t* lds) {
  uint32_t *s_val = lds, *s_piece = lds + REC_NODES * REC_VALS;
  const uint32_t t0 = row * 2 * ROW;
  const uint32_t f = block * 2 * ROW / 21;  // the workgroup's first node, in its row
  const uint32_t ln = threadIdx.x / 3, a = threadIdx.x - 3 * ln;
  const uint32_t t = t0 + f + ln;
  if (threadIdx.x < 192) {  // three waves hold the 3 * REC_NODES threads
    const uint32_t wave_t = t0 + f + (threadIdx.x & ~63u) / 3;
    if (wave_t < A.n_nodes)
      for_segments(A.segs, A.seg_first, A.n_segs, wave_t, t, ln < REC_NODES && t < A.n_nodes,
                   [&](auto* sg, uint32_t d) {
        const bool root = sg->level_kind & SEG_ROOT;
        const K key = A.kl.code(((const K*)sg->elem)[root ? 0u : d >> 3]);
        const K code = root ? key : (key << 3) | (K)(d & 7);
        const float w = sg->width;
        uint32_t* v = s_val + REC_VALS * ln;
        stage_axis(v, a, sg->origin[a] + w * (float)axis_of(code, a), w);
        if (a == 0) v[9] = sg->local0 + d;
      });
  } else if (threadIdx.x - 192 < 21) {
    s_piece[threadIdx.x - 192] = PIECES.slots[threadIdx.x - 192];
  }
  __syncthreads();
#pragma unroll
  for (uint32_t u = 0; u < 2; ++u) {
    const uint32_t p = (2 * block + u) * ROW + threadIdx.x;
    if (t0 + p / 21 < A.n_nodes)
      store_stream((uint4*)A.edges + 21 * (uint64_t)t0 + p, edge_piece(s_val, s_piece, f, p));
  }
}

template <typename K>
__device__ inline void emit_verts(const EmitArgs<K>& A, uint64_t row, uint32_t block) {
  const uint32_t p = block * ROW + threadIdx.x;
  const uint64_t t0 = row * ROW;
  const uint32_t t = (uint32_t)t0 + (p >> 3), wave_t = (uint32_t)t0 + ((p & ~63u) >> 3);
  if (wave_t >= A.n_nodes) return;
  for_segments(A.segs, A.seg_first, A.n_segs, wave_t, t, t < A.n_nodes,
               [&](auto* sg, uint32_t d) {
    store_stream((uint4*)A.verts + 8 * t0 + p, vert_piece(sg->width, p & 7, sg->local0 + d));
  });
}

// Piece q of the voxel codes: the level-1 keys without their mesh bits.
template <typename K>
__device__ inline void emit_voxels(const EmitArgs<K>& A, uint64_t q) {
  if (A.out.code_bytes == 8) {
    const uint64_t i = 2 * q;
    if (i >= A.n_voxels) return;
    const uint64_t c0 = A.kl.code(A.voxels_in[i]);
    const uint64_t c1 = i + 1 < A.n_voxels ? A.kl.code(A.voxels_in[i + 1]) : (K)0;
    store_stream((uint4*)A.voxels + q, make_uint4((uint32_t)c0, (uint32_t)(c0 >> 32),
                                                  (uint32_t)c1, (uint32_t)(c1 >> 32)));
  } else {
    const uint64_t i = 4 * q;
    if (i >= A.n_voxels) return;
    const uint32_t cnt = A.n_voxels - i < 4 ? (uint32_t)(A.n_voxels - i) : 4u;
    K k[4];
    load_consecutive(A.voxels_in + i, ((uintptr_t)A.voxels_in & 15) == 0, cnt, k);
    store_stream((uint4*)A.voxels + q,
                 make_uint4((uint32_t)A.kl.code(k[0]), (uint32_t)A.kl.code(k[1]),
                            (uint32_t)A.kl.code(k[2]), (uint32_t)A.kl.code(k[3])));
  }
}

// Workgroups go round the 8 XCDs in turn.  Of each 128 workgroups of a part
// (of n), XCD x takes 16 consecutive ones, so that the keys that neighboring
// workgroups share are found in its L2 (edge records of 16.1 M nodes: 905 us
// without it, 792 with; the node arrays, whose workgroups share no keys, are
// faster without it).
__device__ inline uint32_t xcd_run(uint32_t b, uint32_t n) {
  return (b | 127u) < n ? (b & ~127u) | ((b & 7u) << 4) | ((b >> 3) & 15u) : b;
}

// Workgroups of each part, in the order they run.
struct EmitBlocks {
  uint32_t nodes, edges, verts, neighbors, voxels;
};

template <typename K>
__global__ __launch_bounds__(ROW) void k_emit(EmitArgs<K> A, EmitBlocks B, uint32_t block0) {
  __shared__ __align__(16) uint32_t lds[8 * ROW + ROW / 4];
  if (A.out.skip && *A.out.skip) return;  // graph replay over changed sizes
  uint32_t b = block0 + blockIdx.x;
  if (b < B.nodes) return emit_nodes(A, b, lds);
  b -= B.nodes;
  if (b < B.edges) b = xcd_run(b, B.edges);
  if (b < B.edges) return emit_edges(A, b / EDGE_BLOCKS, b % EDGE_BLOCKS, lds);
  b -= B.edges;
  if (b < B.verts) return emit_verts(A, b / VERT_BLOCKS, b % VERT_BLOCKS);
  b -= B.verts;
  if (b < B.neighbors) return emit_neighbors(A, (uint64_t)b * ROW + threadIdx.x);
  emit_voxels(A, (uint64_t)(b - B.neighbors) * ROW + threadIdx.x);
}

// The records of nodes that the caller gives: the same pieces from origins
// and widths in memory, one piece a thread.
__global__ __launch_bounds__(ROW) void k_ref_records(const float* origin, const float* width,
                                                     uint64_t n_nodes, uint32_t block0,
                                                     uint32_t edge_blocks, uint32_t* verts,
                                                     uint32_t* edges) {
  __shared__ uint32_t s_val[REC_NODES * REC_VALS], s_piece[21];
  const uint32_t block = block0 + blockIdx.x;
  if (block >= edge_blocks) {
    const uint64_t p = (uint64_t)(block - edge_blocks) * ROW + threadIdx.x, t = p >> 3;
    if (t < n_nodes)
      store_stream((uint4*)verts + p, vert_piece(width[t], p & 7, (uint32_t)t));
    return;
  }
  const uint64_t t0 = (uint64_t)(block / EDGE_BLOCKS) * ROW;
  const uint32_t b = block % EDGE_BLOCKS;
  const uint32_t f = b * ROW / 21, ln = threadIdx.x / 3, a = threadIdx.x - 3 * ln;
  const uint64_t t = t0 + f + ln;
  if (ln < ROW / 21 + 2 && t < n_nodes) {
    stage_axis(s_val + REC_VALS * ln, a, origin[3 * t + a], width[t]);
    if (a == 0) s_val[REC_VALS * ln + 9] = (uint32_t)t;
  }
  if (threadIdx.x < 21) s_piece[threadIdx.x] = PIECES.slots[threadIdx.x];
  __syncthreads();
  const uint32_t p = b * ROW + threadIdx.x;
  if (t0 + p / 21 < n_nodes)
    store_stream((uint4*)edges + 21 * t0 + p, edge_piece(s_val, s_piece, f, p));
}

// ---------------------------------------------------------------- intended neighbors
// Which records a node keeps: bits 0-7 its vertices, 8-19 its edges, 20-25
// its faces (intended semantics).
constexpr uint32_t KEEP_FACES = 20, KEEP_EDGES = 8, KEEP_ALL = (1u << 26) - 1u;

// Neighbor slots of the cells that share corner j (d in {b - 1, b} per axis,
// SVO.cu:567-584), edge i (the two axes that it does not run along take
// {o - 1, o}, SVO.cu:610-627) and face f, without the node's own slot 13.
struct ShareTable {
  uint32_t cells[26];
};
constexpr ShareTable make_share_table() {
  ShareTable t{};
  for (int j = 0; j < 8; ++j)
    for (int q = 0; q < 8; ++q) {
      int slot = 13;
      for (int a = 0, mul = 1; a < 3; ++a, mul *= 3) slot += (((j >> a) & 1) - 1 + ((q >> a) & 1)) * mul;
      t.cells[j] |= 1u << slot;
    }
  for (int i = 0; i < 12; ++i)
    for (int q = 0; q < 4; ++q) {
      int slot = 13, bit = 0;
      for (int a = 0, mul = 1; a < 3; ++a, mul *= 3)
        if (EDGE_ENDS[i][0][a] == EDGE_ENDS[i][1][a])
          slot += ((int)EDGE_ENDS[i][0][a] - 1 + ((q >> bit++) & 1)) * mul;
      t.cells[KEEP_EDGES + i] |= 1u << slot;
    }
  for (int f = 0; f < 6; ++f) t.cells[KEEP_FACES + f] = 1u << FACE_SLOT[f];
  for (int r = 0; r < 26; ++r) t.cells[r] &= ~(1u << 13);
  return t;
}
constexpr ShareTable SHARED = make_share_table();

// Neighbor rows of one level (SVO.cu:522-565 as intended): slot s of child k
// of a group is a child of the parent's neighbor floor((k + d) / 2), child
// (k + d) mod 2 per axis (the closed form of the LUTs, MortonLUT.h:531-597).
// All eight children draw on the parent's 27 neighbors only, and a node's
// children are consecutive, so a workgroup looks up 27 first children per
// group (a thread per node looked up 27 per node: 216 per group, and wrote its
// row with a stride of 108 bytes), builds the rows of 32 groups in LDS and
// writes them, one contiguous run, in 16-byte pieces.  On the way each node's
// records are decided: one is kept by the sharing node of the smallest index
// (`keep`, one word per node, when set), so that the records never read the
// rows again.  2.4 M nodes of the finest level: 940 us before, 86 now.
constexpr uint32_t NB_GROUPS = 32;
__global__ __launch_bounds__(8 * NB_GROUPS) void k_neighbors_level(
    const NodeSeg* segs, const uint32_t* level_segs, const uint32_t* level_blocks,
    uint32_t n_level_segs, int key_bytes, NodeArrays nodes, uint32_t* keep) {
  constexpr uint32_t THREADS = 8 * NB_GROUPS;
  __shared__ uint32_t s_first[NB_GROUPS * 27];
  __shared__ __align__(16) uint32_t s_row[THREADS * 27];
  if (nodes.skip && *nodes.skip) return;  // graph replay over changed sizes
  const uint32_t i = find_seg(level_blocks, n_level_segs, blockIdx.x);
  const auto* sg = scalar_ptr(segs) + scalar_ptr(level_segs)[i];
  const uint32_t kind = sg->level_kind, tid = threadIdx.x;
  if (kind & SEG_ROOT) {  // findNeighbors<true>: the root's own slot alone
    if (tid < 27)
      nodes.neighbors[27 * (uint64_t)sg->t0 + tid] =
          tid == 13 && (kind & 255u) >= 2 ? sg->local0 : NONE;
    if (tid == 0 && keep) keep[sg->t0] = KEEP_ALL;
    return;
  }
  const uint32_t g0 = (blockIdx.x - scalar_ptr(level_blocks)[i]) * NB_GROUPS;
  const uint32_t left = (sg->t1 - sg->t0) / 8 - g0, ng = left < NB_GROUPS ? left : NB_GROUPS;
  const uint64_t base = sg->t0 - sg->local0;  // the mesh's first node
  for (uint32_t x = tid; x < 27 * ng; x += THREADS) {
    const uint32_t gl = x / 27, s = x - 27 * gl, g = g0 + gl;
    uint32_t pn;
    if (kind & SEG_ROOT_CHILD) {
      pn = s == 13 ? sg->parent0 : NONE;
    } else {
      const uint32_t oct = (key_bytes == 8 ? ((const uint32_t*)sg->elem)[2 * (uint64_t)g]
                                           : ((const uint32_t*)sg->elem)[g]) & 7u;
      pn = nodes.neighbors[27 * (base + (sg->parent0 + 8 * sg->group[g] + oct)) + s];
    }
    s_first[x] = pn != NONE ? nodes.childs[8 * (base + pn)] : NONE;
  }
  __syncthreads();
  if (tid < 8 * ng) {
    const uint32_t self = sg->local0 + 8 * g0 + tid;
    // per axis and d = -1, 0, 1: the parent's neighbor and the child in it
    uint32_t off[3][3], ch[3][3];
#pragma unroll
    for (uint32_t a = 0, mul = 1; a < 3; ++a, mul *= 3) {
      const uint32_t bit = (tid >> a) & 1u;
      off[a][0] = (bit - 1) * mul;
      off[a][1] = 0;
      off[a][2] = bit * mul;
      ch[a][0] = ch[a][2] = (bit ^ 1u) << a;
      ch[a][1] = bit << a;
    }
    const uint32_t* first = s_first + 27 * (tid >> 3) + 13;
    uint32_t lower = 0;
#pragma unroll
    for (uint32_t s = 0; s < 27; ++s) {
      const uint32_t x = s % 3, y = s / 3 % 3, z = s / 9;
      const uint32_t f = first[(int32_t)(off[0][x] + off[1][y] + off[2][z])];
      const uint32_t v = f != NONE ? f + (ch[0][x] | ch[1][y] | ch[2][z]) : NONE;
      s_row[27 * tid + s] = v;
      if (v < self) lower |= 1u << s;
    }
    if (keep) {
      uint32_t k = 0;
#pragma unroll
      for (uint32_t r = 0; r < 26; ++r) k |= (lower & SHARED.cells[r]) == 0 ? 1u << r : 0u;
      keep[sg->t0 + 8 * g0 + tid] = k;
    }
  }
  __syncthreads();
  // the rows, 216 * ng words from a 4-byte boundary; the finest level's go past
  // the caches, the others the next level reads (96 -> 86 us for the finest of
  // 2.4 M nodes; 104 when its own rows stay in the caches as well)
  const uint64_t w0 = 27 * ((uint64_t)sg->t0 + 8 * g0);
  write_words(
      nodes.neighbors, w0, 216 * ng, tid, THREADS, [&](uint32_t i) { return s_row[i]; },
      (kind & 255u) == 1);
}

// ---------------------------------------------------------------- kept records
// Records by keep masks: count per block of KEEP_BLOCK nodes, scan, write.

// Reference semantics when a record may equal its predecessor, which drops it
// (uniqueVert / uniqueEdge, SVO.cu:679-720): a node's vertices and edges
// against their predecessors, the last of them the previous node's.
__global__ __launch_bounds__(ROW) void k_ref_keep(NodeArrays nodes, uint64_t n_nodes,
                                                  const NodeSeg* segs, const uint32_t* seg_first,
                                                  uint32_t n_segs, uint32_t* keep) {
  if (nodes.skip && *nodes.skip) return;  // graph replay over changed sizes
  const uint32_t t = blockIdx.x * ROW + threadIdx.x;
  if ((t & ~63u) >= n_nodes) return;
  for_segments(segs, seg_first, n_segs, t & ~63u, t, t < n_nodes, [&](auto* sg, uint32_t d) {
    const bool first = sg->local0 + d == 0;
    const NodeGeom g = load_geom(nodes, t), gp = first ? g : load_geom(nodes, t - 1);
    uint32_t k = 0;
    float prev[3], p[3], pa[3], pb[3], a[3], b[3];
    ref_corner(gp.w, 7, prev);
    for (int j = 0; j < 8; ++j) {
      ref_corner(g.w, j, p);
      if ((j == 0 && first) || !eq3(p, prev)) k |= 1u << j;
      for (int q = 0; q < 3; ++q) prev[q] = p[q];
    }
    ref_edge(gp, 11, pa, pb);
    for (int i = 0; i < 12; ++i) {
      ref_edge(g, i, a, b);
      if ((i == 0 && first) || !edge_eq(a, b, pa, pb)) k |= 1u << (KEEP_EDGES + i);
      for (int q = 0; q < 3; ++q) {
        pa[q] = a[q];
        pb[q] = b[q];
      }
    }
    keep[t] = k;
  });
}

__device__ inline void keep_counts(uint32_t k, uint32_t& v, uint32_t& e, uint32_t& f) {
  v = __popc(k & 0xFFu);
  e = __popc((k >> KEEP_EDGES) & 0xFFFu);
  f = __popc(k >> KEEP_FACES);
}

// One wave per block of KEEP_BLOCK nodes: counts[{v, e, f} * n_blocks + block].
constexpr uint32_t KEEP_BLOCK = 512;
__global__ __launch_bounds__(BLOCK) void k_keep_count(const uint32_t* keep, uint64_t n_nodes,
                                                      uint32_t n_blocks, uint32_t* counts,
                                                      const uint32_t* skip) {
  if (skip && *skip) return;  // graph replay over changed sizes
  const uint64_t block = (uint64_t)blockIdx.x * (BLOCK / 64) + (threadIdx.x >> 6);
  if (block * KEEP_BLOCK >= n_nodes) return;
  uint32_t sv = 0, se = 0, sf = 0;
#pragma unroll
  for (uint32_t u = 0; u < KEEP_BLOCK / 64; ++u) {
    const uint64_t t = block * KEEP_BLOCK + u * 64 + __lane_id();
    uint32_t v, e, f;
    keep_counts(t < n_nodes ? keep[t] : 0u, v, e, f);
    sv += v;
    se += e;
    sf += f;
  }
  sv = wave_sum_u32(sv);
  se = wave_sum_u32(se);
  sf = wave_sum_u32(sf);
  if (__lane_id() == 0) {
    counts[block] = sv;
    counts[n_blocks + block] = se;
    counts[2 * (uint64_t)n_blocks + block] = sf;
  }
}

// Exclusive sums of the block counts and the totals: a workgroup per kind, four
// rounds' loads in flight (one workgroup for all kinds, a round at a time: 12
// us for 6382 blocks, 5 so).
constexpr uint32_t KEEP_SCAN = 1024, KEEP_AHEAD = 4;
__global__ __launch_bounds__(KEEP_SCAN) void k_keep_scan(const uint32_t* counts, uint32_t n_blocks,
                                                         uint64_t* offsets,
                                                         unsigned long long* totals,
                                                         const uint32_t* skip) {
  if (skip && *skip) return;  // graph replay over changed sizes
  __shared__ uint32_t s_wave[KEEP_AHEAD][KEEP_SCAN / 64];
  const uint32_t* in = counts + (uint64_t)blockIdx.x * n_blocks;
  uint64_t* out = offsets + (uint64_t)blockIdx.x * n_blocks;
  uint64_t carry = 0;
  const uint32_t wave = threadIdx.x >> 6;
  for (uint32_t b0 = 0; b0 < n_blocks; b0 += KEEP_SCAN * KEEP_AHEAD) {
    uint32_t c[KEEP_AHEAD], inc[KEEP_AHEAD];
#pragma unroll
    for (uint32_t j = 0; j < KEEP_AHEAD; ++j) {
      const uint32_t b = b0 + j * KEEP_SCAN + threadIdx.x;
      c[j] = b < n_blocks ? in[b] : 0u;
    }
#pragma unroll
    for (uint32_t j = 0; j < KEEP_AHEAD; ++j) {
      inc[j] = wave_incl_scan_dpp(c[j]);  // at most 1024 * 6144 over the workgroup
      if ((threadIdx.x & 63) == 63) s_wave[j][wave] = inc[j];
    }
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < KEEP_AHEAD; ++j) {
      uint32_t pre = 0, all = 0;
      for (uint32_t w = 0; w < KEEP_SCAN / 64; ++w) {
        const uint32_t x = s_wave[j][w];
        if (w < wave) pre += x;
        all += x;
      }
      const uint32_t b = b0 + j * KEEP_SCAN + threadIdx.x;
      if (b < n_blocks) out[b] = carry + pre + inc[j] - c[j];
      carry += all;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) totals[blockIdx.x] = carry;
}

// Coordinates of the records in order, two bits each: 0 the node's origin bare
// (an end without offset), 1 origin + 0, 2 origin + width.
struct WordTable {
  uint16_t edge[12], face[6], vert[8];
};
constexpr WordTable make_word_table() {
  WordTable t{};
  auto term = [](const uint8_t(&e)[3], int a) {
    return !e[0] && !e[1] && !e[2] ? 0 : e[a] ? 2 : 1;
  };
  for (int w = 0; w < 6; ++w) {
    for (int i = 0; i < 12; ++i) t.edge[i] |= (uint16_t)(term(EDGE_ENDS[i][w / 3], w % 3) << 2 * w);
    for (int f = 0; f < 6; ++f) t.face[f] |= (uint16_t)(term(FACE_ENDS[f][w / 3], w % 3) << 2 * w);
  }
  for (int j = 0; j < 8; ++j) {
    const uint8_t corner[3] = {(uint8_t)(j & 1), (uint8_t)(j >> 1 & 1), (uint8_t)(j >> 2 & 1)};
    for (int a = 0; a < 3; ++a) t.vert[j] |= (uint16_t)(term(corner, a) << 2 * a);
  }
  return t;
}
__constant__ WordTable WORDS = make_word_table();

// Writes one kind of the kept records of a block of nodes (grid: the blocks'
// vertices, then their edges, then their faces, so that the stores in flight
// lie close together): the nodes' values, from the level's keys as in the
// emission, and the list of kept records (node and record, in order) are
// staged in LDS; then a thread looks up a record's words, and the array's run
// of words is written in 16-byte pieces from LDS, a wave's 1024 bytes from the
// start of a cache line.  3.3 M nodes, 792 MB: 160 us (172 with waves that
// begin anywhere; 190 a word at a time from the list, bound by instructions),
// and 5 for the count.  (A thread per node that wrote its own records
// scattered 16- and 28-byte stores, after deciding twice from its neighbor row
// which they are: 1,240 and 300 for the count.)
template <typename K>
__global__ __launch_bounds__(KEEP_BLOCK) void k_keep_write(
    bool reference, KeyLayout<K> kl, NodeArrays nodes, uint64_t n_nodes, uint32_t n_blocks,
    const NodeSeg* segs, const uint32_t* seg_first, uint32_t n_segs, const uint32_t* keep,
    const uint64_t* offsets, AttrOut out) {
  if (nodes.skip && *nodes.skip) return;  // graph replay over changed sizes
  constexpr uint32_t VALS = 5;  // origin, width, owner
  __shared__ uint32_t s_val[KEEP_BLOCK * VALS];
  __shared__ __align__(16) uint32_t s_stage[7 * KEEP_BLOCK + 4];
  __shared__ uint16_t s_list[KEEP_BLOCK * 12];
  __shared__ uint32_t s_word[12];
  __shared__ uint32_t s_sum[KEEP_BLOCK / 64];
  const uint32_t what = blockIdx.x / n_blocks, block = blockIdx.x - what * n_blocks;
  const uint32_t tid = threadIdx.x, t = block * KEEP_BLOCK + tid;
  if (tid < 12)
    s_word[tid] = what == 1 ? WORDS.edge[tid] : what == 2 ? WORDS.face[tid % 6] : WORDS.vert[tid & 7];
  const uint32_t all = t < n_nodes ? keep[t] : 0u;
  const uint32_t bits = what == 0   ? all & 0xFFu
                        : what == 1 ? all >> KEEP_EDGES & 0xFFFu
                                    : all >> KEEP_FACES;
  // exclusive sums over the block
  const uint32_t inc = wave_incl_scan_dpp(__popc(bits));
  if ((tid & 63) == 63) s_sum[tid >> 6] = inc;
  __syncthreads();
  uint32_t count = 0, at = inc - __popc(bits);
#pragma unroll
  for (uint32_t w = 0; w < KEEP_BLOCK / 64; ++w) {
    if (w < tid >> 6) at += s_sum[w];
    count += s_sum[w];
  }
  const uint64_t first = offsets[blockIdx.x];
  if ((t & ~63u) < n_nodes)
    for_segments(segs, seg_first, n_segs, t & ~63u, t, t < n_nodes, [&](auto* sg, uint32_t d) {
      // origin and width from the level's keys, as emit_nodes has them
      const uint32_t local = sg->local0 + d;
      const float w = sg->width;
      const K* elem = (const K*)sg->elem;
      const K code = sg->level_kind & SEG_ROOT ? kl.code(elem[0])
                                               : (K)((kl.code(elem[d >> 3]) << 3) | (K)(d & 7));
      uint32_t* v = s_val + VALS * tid;
#pragma unroll
      for (uint32_t x = 0; x < 3; ++x)
        v[x] = __float_as_uint(sg->origin[x] + w * (float)axis_of(code, x));
      v[3] = __float_as_uint(w);
      v[4] = local;
      if (local == 0) out.totals[4 + 3 * sg->mesh + what] = first + at;
    });
  for (uint32_t r = bits, i = at; r; r &= r - 1u)
    s_list[i++] = (uint16_t)((tid << 4) | __builtin_ctz(r));
  __syncthreads();
  // word j < 3 k of a record: its coordinate's term of that axis
  struct Node {
    float term[3][3];
    uint32_t owner;
  };
  auto node_of = [&](uint32_t e) {
    const uint32_t* v = s_val + VALS * (e >> 4);
    const float w = __uint_as_float(v[3]);
    Node n;
#pragma unroll
    for (uint32_t x = 0; x < 3; ++x) {
      const float o = __uint_as_float(v[x]);
      n.term[0][x] = o;
      n.term[1][x] = o + 0.0f;
      n.term[2][x] = o + w;
      if (what == 0 && reference) {  // the reference's vertices have no origin
        n.term[0][x] = n.term[1][x] = w * 0.0f;
        n.term[2][x] = w * 1.0f;
      }
    }
    n.owner = v[4];
    return n;
  };
  auto coord = [](const Node& n, uint32_t word, uint32_t j) {
    const uint32_t k = word >> 2 * j & 3u, x = j % 3;
    const uint32_t a = __float_as_uint(n.term[0][x]), b = __float_as_uint(n.term[1][x]),
                   c = __float_as_uint(n.term[2][x]);
    return k == 0 ? a : k == 1 ? b : c;
  };
  if (what == 0) {  // a vertex is a piece
    for (uint32_t r = tid; r < count; r += KEEP_BLOCK) {
      const uint32_t e = s_list[r], w = s_word[e & 15u];
      const Node n = node_of(e);
      store_stream((uint4*)out.verts + first + r,
                   make_uint4(coord(n, w, 0), coord(n, w, 1), coord(n, w, 2), n.owner));
    }
    return;
  }
  // edges and faces, KEEP_BLOCK at a time
  uint32_t* dst = (uint32_t*)(what == 1 ? out.edges : out.faces);
  for (uint32_t c = 0; c < count; c += KEEP_BLOCK) {
    const uint32_t k = count - c < KEEP_BLOCK ? count - c : KEEP_BLOCK;
    const uint64_t w0 = 7 * (first + c);
    uint32_t* stage = s_stage + (w0 & 3u);
    if (tid < k) {
      const uint32_t e = s_list[c + tid], w = s_word[e & 15u];
      const Node n = node_of(e);
#pragma unroll
      for (uint32_t j = 0; j < 6; ++j) stage[7 * tid + j] = coord(n, w, j);
      stage[7 * tid + 6] = n.owner;
    }
    __syncthreads();
    write_words(
        dst, w0, 7 * k, tid, KEEP_BLOCK, [&](uint32_t i) { return stage[i]; },
        [&](uint32_t i) { return *(const uint4*)(stage + i); });
    __syncthreads();
  }
}

// 168-byte SVONode records (SVO.h:20-35), one thread per 32-bit word.
__global__ void k_pack_aos(NodeArrays n, uint64_t first, uint64_t count, uint32_t* dst) {
  const uint64_t gid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= count * 42) return;
  const uint64_t r = gid / 42;
  const uint32_t wd = (uint32_t)(gid - r * 42);
  const uint64_t t = first + r;
  uint32_t v;
  if (wd == 0) v = n.code_bytes == 8 ? (uint32_t)((const uint64_t*)n.code)[t]
                                     : ((const uint32_t*)n.code)[t];
  else if (wd == 1) v = n.is_leaf[t];  // bool + three zero padding bytes
  else if (wd < 5) v = __float_as_uint(n.origin[3 * t + (wd - 2)]);
  else if (wd == 5) v = __float_as_uint(n.width[t]);
  else if (wd == 6) v = n.parent[t];
  else if (wd < 15) v = n.childs[8 * t + (wd - 7)];
  else v = n.neighbors[27 * t + (wd - 15)];
  dst[gid] = v;
}

__global__ void k_query(const uint32_t* nb, uint64_t n_nodes, const uint32_t* node,
                        const uint8_t* slot, uint64_t n, uint32_t* out) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t t = node[i];
  const uint32_t s = slot[i];
  out[i] = (t < n_nodes && s < 27) ? nb[27 * (uint64_t)t + s] : NONE;
}

// At most RING_BLOCKS workgroups; bound by the two trips over the link to the host.
constexpr int QUERY_THREADS = 1024;
__global__ __launch_bounds__(QUERY_THREADS) void k_query_ring(const uint32_t* nb, uint64_t n_nodes,
                                                              const uint32_t* node,
                                                              const uint8_t* slot, uint64_t n,
                                                              uint32_t* out, uint32_t* flags,
                                                              uint32_t number) {
  constexpr int AHEAD = 4;
  const uint64_t step = (uint64_t)gridDim.x * QUERY_THREADS;
  for (uint64_t i = (uint64_t)blockIdx.x * QUERY_THREADS + threadIdx.x; i < n; i += AHEAD * step) {
    uint32_t t[AHEAD], v[AHEAD];
    uint8_t s[AHEAD];
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) {
      const bool in = i + j * step < n;
      t[j] = in ? node[i + j * step] : NONE;
      s[j] = in ? slot[i + j * step] : 27;
    }
#pragma unroll
    for (int j = 0; j < AHEAD; ++j)
      v[j] = t[j] < n_nodes && s[j] < 27 ? nb[27 * (uint64_t)t[j] + s[j]] : NONE;
#pragma unroll
    for (int j = 0; j < AHEAD; ++j)
      if (i + j * step < n) out[i + j * step] = v[j];
  }
  __threadfence_system();
  __syncthreads();
  if (threadIdx.x == 0)
    __hip_atomic_store(flags + blockIdx.x, number, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

inline uint32_t grid_for(uint64_t threads) { return (uint32_t)((threads + BLOCK - 1) / BLOCK); }

}  // namespace

template <typename K>
void launch_emit(const EmitArgs<K>& a, hipStream_t s) {
  const uint32_t rows = (uint32_t)((a.n_nodes + ROW - 1) / ROW);
  auto blocks = [](uint64_t words) { return (uint32_t)(((words + 3) / 4 + ROW - 1) / ROW); };
  const EmitBlocks b{rows, a.records ? EDGE_BLOCKS * ((rows + 1) / 2) : 0,
                     a.records ? VERT_BLOCKS * rows : 0,
                     a.neighbors ? blocks(27 * a.n_nodes) : 0,
                     blocks(a.n_voxels * (uint64_t)(a.out.code_bytes / 4))};
  const uint32_t n = b.nodes + b.edges + b.verts + b.neighbors + b.voxels;
  for (uint32_t b0 = 0; b0 < n; b0 += BLOCKS_PER_LAUNCH)
    hipLaunchKernelGGL(k_emit<K>, dim3(std::min(n - b0, BLOCKS_PER_LAUNCH)),
                       dim3(ROW), 0, s, a, b, b0);
  if (a.neighbors && a.n_roots > 1)
    hipLaunchKernelGGL(k_root_slots, dim3((a.n_segs + 63) / 64), dim3(64), 0, s, a.segs, a.n_segs,
                       a.out);
}

// RING_BLOCKS workgroups take a part of each piece, in the pieces' order, so
// that the first pieces arrive while the later ones are on their way.  Bound
// by the link to the host.
template <typename W>
__device__ inline void copy_part(const char* src, char* dst, uint64_t bytes) {
  constexpr int AHEAD = 4;
  const uint64_t n = bytes / sizeof(W), step = (uint64_t)RING_BLOCKS * BLOCK;
  for (uint64_t i = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; i < n; i += AHEAD * step) {
    W w[AHEAD];
#pragma unroll
    for (int j = 0; j < AHEAD; ++j)
      if (i + j * step < n) w[j] = ((const W*)src)[i + j * step];
#pragma unroll
    for (int j = 0; j < AHEAD; ++j)
      if (i + j * step < n) ((W*)dst)[i + j * step] = w[j];
  }
  // the bytes behind the last whole word
  if (blockIdx.x == 0 && threadIdx.x < bytes - n * sizeof(W))
    dst[n * sizeof(W) + threadIdx.x] = src[n * sizeof(W) + threadIdx.x];
}
__global__ __launch_bounds__(BLOCK) void k_ring_copy(const char* src, uint64_t bytes, char* ring,
                                                     uint32_t* flags, uint64_t slot,
                                                     uint32_t number) {
  for (uint64_t at = 0; at < bytes; at += RING_PIECE, slot = (slot + 1) % RING_SLOTS) {
    const uint64_t k = bytes - at < RING_PIECE ? bytes - at : RING_PIECE;
    char* dst = ring + slot * RING_PIECE;
    if (((uintptr_t)src & 15) == 0) copy_part<uint4>(src + at, dst, k);
    else if (((uintptr_t)src & 3) == 0) copy_part<uint32_t>(src + at, dst, k);
    else copy_part<uint8_t>(src + at, dst, k);
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0)
      __hip_atomic_store(flags + slot * RING_BLOCKS + blockIdx.x, number, __ATOMIC_RELEASE,
                         __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

__global__ void k_copy_u32(uint32_t* dst, const uint32_t* src, uint64_t n) {
  for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    dst[i] = src[i];
}

// Sets *flag when any of the n words differs from its expected value.
__global__ void k_check_equal(const uint32_t* got, const uint32_t* want, uint64_t n,
                              uint32_t* flag) {
  uint32_t diff = 0;
  for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    diff |= got[i] ^ want[i];
  if (__any(diff != 0) && (threadIdx.x & 63) == 0) atomicOr(flag, 1u);
}

void launch_check_equal(const void* got, const void* want, uint64_t bytes, uint32_t* flag,
                        hipStream_t s) {
  const uint64_t n = bytes / 4;
  if (n == 0) return;
  const uint64_t blocks = std::min<uint64_t>((n + BLOCK - 1) / BLOCK, 256);
  hipLaunchKernelGGL(k_check_equal, dim3((uint32_t)blocks), dim3(BLOCK), 0, s,
                     (const uint32_t*)got, (const uint32_t*)want, n, flag);
}

hipError_t launch_ring_copy(const void* src, uint64_t bytes, void* ring, uint32_t* flags,
                            uint64_t slot, uint32_t number, hipStream_t s) {
  void* args[] = {&src, &bytes, &ring, &flags, &slot, &number};
  return hipLaunchKernel((const void*)k_ring_copy, dim3(RING_BLOCKS), dim3(BLOCK), args, 0, s);
}

void launch_copy_u32(uint32_t* dst, const uint32_t* src, uint64_t n, hipStream_t s) {
  if (n == 0) return;
  const uint64_t blocks = std::min<uint64_t>((n + BLOCK - 1) / BLOCK, 256);
  hipLaunchKernelGGL(k_copy_u32, dim3((uint32_t)blocks), dim3(BLOCK), 0, s, dst, src, n);
}

void launch_fill_u32(uint32_t* p, uint32_t value, uint64_t n, hipStream_t s) {
  if (n == 0) return;
  const uint64_t blocks = std::min<uint64_t>(grid_for((n + 3) / 4), 1u << 20);
  hipLaunchKernelGGL(k_fill_u32, dim3((uint32_t)blocks), dim3(BLOCK), 0, s, p, value, n);
}

void launch_neighbors_level(const NodeSeg* segs, const uint32_t* level_segs,
                            const uint32_t* level_blocks, uint32_t n_level_segs, uint32_t blocks,
                            int key_bytes, NodeArrays nodes, uint32_t* keep, hipStream_t s) {
  if (blocks == 0) return;
  hipLaunchKernelGGL(k_neighbors_level, dim3(blocks), dim3(8 * NB_GROUPS), 0, s, segs, level_segs,
                     level_blocks, n_level_segs, key_bytes, nodes, keep);
}

uint32_t neighbor_blocks(const NodeSeg& seg) {
  return seg.level_kind & SEG_ROOT ? 1u : ((seg.t1 - seg.t0) / 8 + NB_GROUPS - 1) / NB_GROUPS;
}

// keep masks, then per block of nodes the counts (padded to 8 bytes) and offsets
static uint64_t keep_blocks(uint64_t n_nodes) { return (n_nodes + KEEP_BLOCK - 1) / KEEP_BLOCK; }
size_t keep_bytes(uint64_t n_nodes) {
  return (size_t)(4 * KEEP_BLOCK + 16 + 24) * keep_blocks(n_nodes);
}

template <typename K>
void launch_kept_records(int semantics, KeyLayout<K> kl, const NodeArrays& nodes, uint64_t n_nodes,
                         const NodeSeg* segs, const uint32_t* seg_first, uint32_t n_segs,
                         void* tmp, AttrOut out, hipStream_t s) {
  const uint32_t nb = (uint32_t)keep_blocks(n_nodes);
  uint32_t* keep = (uint32_t*)tmp;
  uint64_t* offsets = (uint64_t*)(keep + (uint64_t)KEEP_BLOCK * nb);
  uint32_t* counts = (uint32_t*)(offsets + 3 * (uint64_t)nb);
  const bool reference = semantics == SVO_SEM_REFERENCE;
  if (reference)
    hipLaunchKernelGGL(k_ref_keep, dim3((uint32_t)((n_nodes + ROW - 1) / ROW)), dim3(ROW), 0, s,
                       nodes, n_nodes, segs, seg_first, n_segs, keep);
  hipLaunchKernelGGL(k_keep_count, dim3((nb + 3) / 4), dim3(BLOCK), 0, s, (const uint32_t*)keep,
                     n_nodes, nb, counts, nodes.skip);
  hipLaunchKernelGGL(k_keep_scan, dim3(3), dim3(KEEP_SCAN), 0, s, (const uint32_t*)counts, nb,
                     offsets, out.totals, nodes.skip);
  hipLaunchKernelGGL(k_keep_write<K>, dim3(reference ? 2 * nb : 3 * nb), dim3(KEEP_BLOCK), 0, s,
                     reference, kl, nodes, n_nodes, nb, segs, seg_first, n_segs,
                     (const uint32_t*)keep, (const uint64_t*)offsets, out);
}

void launch_ref_records(const float* origin, const float* width, uint64_t n_nodes,
                        svo_vertex_t* verts, svo_edge_t* edges, hipStream_t s) {
  const uint32_t rows = (uint32_t)((n_nodes + ROW - 1) / ROW);
  const uint32_t n = rows * (EDGE_BLOCKS + VERT_BLOCKS);
  for (uint32_t b0 = 0; b0 < n; b0 += BLOCKS_PER_LAUNCH)
    hipLaunchKernelGGL(k_ref_records, dim3(std::min(n - b0, BLOCKS_PER_LAUNCH)), dim3(ROW), 0, s,
                       origin, width, n_nodes, b0, rows * EDGE_BLOCKS, (uint32_t*)verts,
                       (uint32_t*)edges);
}

void launch_pack_aos(const NodeArrays& nodes, uint64_t first, uint64_t n, void* dst,
                     hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_pack_aos, dim3(grid_for(42 * n)), dim3(BLOCK), 0, s, nodes, first, n,
                     (uint32_t*)dst);
}

void launch_query_neighbors(const uint32_t* neighbors, uint64_t n_nodes, const uint32_t* node,
                            const uint8_t* slot, uint64_t n, uint32_t* out, hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_query, dim3(grid_for(n)), dim3(BLOCK), 0, s, neighbors, n_nodes, node,
                     slot, n, out);
}

uint32_t query_ring_blocks(uint64_t n) {
  return (uint32_t)std::min<uint64_t>((n + QUERY_THREADS - 1) / QUERY_THREADS, RING_BLOCKS);
}
hipError_t launch_query_ring(const uint32_t* neighbors, uint64_t n_nodes, const uint32_t* node,
                             const uint8_t* slot, uint64_t n, uint32_t* out, uint32_t* flags,
                             uint32_t number, hipStream_t s) {
  void* args[] = {&neighbors, &n_nodes, &node, &slot, &n, &out, &flags, &number};
  return hipLaunchKernel((const void*)k_query_ring, dim3(query_ring_blocks(n)),
                         dim3(QUERY_THREADS), args, 0, s);
}

template void launch_kept_records<uint32_t>(int, KeyLayout<uint32_t>, const NodeArrays&, uint64_t,
                                            const NodeSeg*, const uint32_t*, uint32_t, void*,
                                            AttrOut, hipStream_t);
template void launch_kept_records<uint64_t>(int, KeyLayout<uint64_t>, const NodeArrays&, uint64_t,
                                            const NodeSeg*, const uint32_t*, uint32_t, void*,
                                            AttrOut, hipStream_t);
template void launch_emit<uint32_t>(const EmitArgs<uint32_t>&, hipStream_t);
template void launch_emit<uint64_t>(const EmitArgs<uint64_t>&, hipStream_t);

}  // namespace svo
