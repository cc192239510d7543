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
// index.  Count -> scan -> write, node-major.
#include <algorithm>

#include "svo_internal.h"
#include "svo_scan.h"

namespace svo {
namespace {

constexpr int BLOCK = 256;

// Node (group g at `level`, child key k) of the neighbor kernel.
template <typename K>
struct GroupNode {
  bool live;
  uint32_t m;
  K P;            // parent key (element g of the next level)
  uint64_t local; // node index within its mesh
  uint32_t parent;
};

template <typename K>
__device__ inline GroupNode<K> group_node(int level, KeyLayout<K> kl, const K* elem_next,
                                          const uint32_t* group_next, uint64_t n_groups,
                                          const LevelSpan* spans, uint32_t n_levels,
                                          const MeshTreeState* state,
                                          const MeshNodeLayout* layout, uint64_t g, uint32_t k) {
  GroupNode<K> r;
  r.live = false;
  r.m = 0;
  r.P = 0;
  r.local = 0;
  r.parent = NONE;
  if (g >= n_groups) return r;
  r.P = elem_next[g];
  r.m = kl.mesh(r.P);
  const uint32_t depth = state[r.m].depth;
  if (depth <= (uint32_t)level) return r;  // depth-1 tree: its level-1 group is not a node group
  const MeshNodeLayout& L = layout[r.m];
  if (L.n_nodes == 0) return r;  // mesh rejected after the level phase
  r.live = true;
  const LevelSpan sp = spans[(uint64_t)r.m * n_levels + (level - 1)];
  r.local = L.level_off[level - 1] + 8ull * (g - sp.group_first) + k;
  if (depth == (uint32_t)level + 1) {
    r.parent = (uint32_t)L.level_off[level];  // the root
  } else {
    const LevelSpan spn = spans[(uint64_t)r.m * n_levels + level];
    r.parent = (uint32_t)(L.level_off[level] + 8ull * (group_next[g] - spn.group_first) +
                          (uint32_t)(r.P & 7));
  }
  return r;
}

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

// Neighbor LUTs (MortonLUT.h:531-597) in closed form: slot s = (dx+1) +
// 3(dy+1) + 9(dz+1); child k's neighbor in direction d is child
// ((k+d) mod 2 per axis) of the parent-level neighbor floor((k+d)/2).
__device__ inline void nb_lut(uint32_t k, uint32_t s, uint32_t& pslot, uint32_t& child) {
  const int d[3] = {(int)(s % 3) - 1, (int)((s / 3) % 3) - 1, (int)(s / 9) - 1};
  const int mul[3] = {1, 3, 9};
  int ps = 0, ch = 0;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const int c = (int)((k >> a) & 1u) + d[a];
    const int p = c < 0 ? -1 : (c >> 1);
    ps += (p + 1) * mul[a];
    ch |= (c & 1) << a;
  }
  pslot = (uint32_t)ps;
  child = (uint32_t)ch;
}

template <typename K>
__global__ __launch_bounds__(BLOCK) void k_neighbors_level(
    int level, KeyLayout<K> kl, const K* elem_next, const uint32_t* group_next,
    uint64_t n_groups, const LevelSpan* spans, uint32_t n_levels, const MeshTreeState* state,
    const MeshNodeLayout* layout, NodeArrays nodes) {
  if (nodes.skip && *nodes.skip) return;  // graph replay over changed sizes
  const uint64_t gid = (uint64_t)blockIdx.x * BLOCK + threadIdx.x;
  const uint64_t g = gid >> 3;
  const uint32_t k = (uint32_t)(gid & 7);
  const GroupNode<K> gn = group_node(level, kl, elem_next, group_next, n_groups, spans, n_levels,
                                     state, layout, g, k);
  if (!gn.live) return;
  const uint64_t base = layout[gn.m].node_base;
  const uint32_t* pn_row = nodes.neighbors + 27 * (base + gn.parent);
  uint32_t* row = nodes.neighbors + 27 * (base + gn.local);
  for (uint32_t s = 0; s < 27; ++s) {
    uint32_t ps, ch;
    nb_lut(k, s, ps, ch);
    const uint32_t pn = pn_row[ps];
    row[s] = pn != NONE ? nodes.childs[8 * (base + pn) + ch] : NONE;
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
__constant__ uint8_t FACE_OFS[6][2][3] = {{{0, 0, 0}, {0, 1, 1}}, {{1, 0, 0}, {1, 1, 1}},
                                          {{0, 0, 0}, {1, 0, 1}}, {{0, 1, 0}, {1, 1, 1}},
                                          {{0, 0, 0}, {1, 1, 0}}, {{0, 0, 1}, {1, 1, 1}}};
__constant__ uint8_t FACE_SLOT[6] = {12, 14, 10, 16, 4, 22};

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

// Cells sharing corner j: d in {b-1, b} per axis, x fastest (SVO.cu:567-584).
__device__ inline uint32_t vert_slot(int j, int q) {
  const int dx = ((j >> 0) & 1) - 1 + ((q >> 0) & 1);
  const int dy = ((j >> 1) & 1) - 1 + ((q >> 1) & 1);
  const int dz = ((j >> 2) & 1) - 1 + ((q >> 2) & 1);
  return (uint32_t)((dx + 1) + 3 * (dy + 1) + 9 * (dz + 1));
}
// Cells sharing edge i: the two axes the edge does not run along take
// {o-1, o}; the running axis takes 0 (SVO.cu:610-627).
__device__ inline uint32_t edge_slot(int i, int q) {
  const uint8_t* a = EDGE_OFS[i][0];
  const uint8_t* b = EDGE_OFS[i][1];
  int d[3];
  int bitpos = 0;
  for (int ax = 0; ax < 3; ++ax) {
    if (a[ax] != b[ax]) {
      d[ax] = 0;
    } else {
      d[ax] = (int)a[ax] - 1 + ((q >> bitpos) & 1);
      ++bitpos;
    }
  }
  return (uint32_t)((d[0] + 1) + 3 * (d[1] + 1) + 9 * (d[2] + 1));
}

__device__ inline uint32_t find_mesh64(const uint64_t* base, uint32_t n_meshes, uint64_t t) {
  uint32_t lo = 0, hi = n_meshes;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (base[mid] <= t) lo = mid; else hi = mid;
  }
  return lo;
}

struct AttrCounts {
  uint32_t v, e, f;
};

// Counts (and optionally writes) the records of node t.
template <bool WRITE>
__device__ inline AttrCounts node_attrs(int semantics, const NodeArrays& n, uint64_t t,
                                        uint64_t local, uint64_t vpos, uint64_t epos,
                                        uint64_t fpos, AttrOut out) {
  AttrCounts c = {0, 0, 0};
  const NodeGeom g = load_geom(n, t);
  const uint32_t self = (uint32_t)local;
  if (semantics == SVO_SEM_REFERENCE) {
    float prev[3];
    if (local > 0) ref_corner(n.width[t - 1], 7, prev);
    for (int j = 0; j < 8; ++j) {
      float p[3];
      ref_corner(g.w, j, p);
      const bool keep = (j == 0 && local == 0) || !eq3(p, prev);
      if (keep) {
        if (WRITE) {
          svo_vertex_t r;
          r.p[0] = p[0];
          r.p[1] = p[1];
          r.p[2] = p[2];
          r.owner = self;
          out.verts[vpos + c.v] = r;
        }
        ++c.v;
      }
      prev[0] = p[0];
      prev[1] = p[1];
      prev[2] = p[2];
    }
    float pa[3], pb[3];
    if (local > 0) {
      const NodeGeom gp = load_geom(n, t - 1);
      ref_edge(gp, 11, pa, pb);
    }
    for (int i = 0; i < 12; ++i) {
      float a[3], b[3];
      ref_edge(g, i, a, b);
      const bool keep = (i == 0 && local == 0) || !edge_eq(a, b, pa, pb);
      if (keep) {
        if (WRITE) {
          svo_edge_t r;
          for (int q = 0; q < 3; ++q) {
            r.a[q] = a[q];
            r.b[q] = b[q];
          }
          r.owner = self;
          out.edges[epos + c.e] = r;
        }
        ++c.e;
      }
      for (int q = 0; q < 3; ++q) {
        pa[q] = a[q];
        pb[q] = b[q];
      }
    }
    return c;
  }
  const uint32_t* nb = n.neighbors + 27 * t;
  for (int j = 0; j < 8; ++j) {
    uint32_t owner = self;
    for (int q = 0; q < 8; ++q) {
      const uint32_t v = nb[vert_slot(j, q)];
      owner = v < owner ? v : owner;
    }
    if (owner != self) continue;
    if (WRITE) {
      const uint8_t ofs[3] = {(uint8_t)(j & 1), (uint8_t)((j >> 1) & 1), (uint8_t)((j >> 2) & 1)};
      svo_vertex_t r;
      offset_point(g.o, g.w, ofs, r.p);
      r.owner = self;
      out.verts[vpos + c.v] = r;
    }
    ++c.v;
  }
  for (int i = 0; i < 12; ++i) {
    uint32_t owner = self;
    for (int q = 0; q < 4; ++q) {
      const uint32_t v = nb[edge_slot(i, q)];
      owner = v < owner ? v : owner;
    }
    if (owner != self) continue;
    if (WRITE) {
      svo_edge_t r;
      ref_edge(g, i, r.a, r.b);
      r.owner = self;
      out.edges[epos + c.e] = r;
    }
    ++c.e;
  }
  for (int f = 0; f < 6; ++f) {
    const uint32_t v = nb[FACE_SLOT[f]];
    if (v < self) continue;
    if (WRITE) {
      svo_edge_t r;
      offset_point(g.o, g.w, FACE_OFS[f][0], r.a);
      offset_point(g.o, g.w, FACE_OFS[f][1], r.b);
      r.owner = self;
      out.faces[fpos + c.f] = r;
    }
    ++c.f;
  }
  return c;
}

__device__ inline void block_range(uint64_t n, uint32_t G, uint32_t b, uint64_t& beg,
                                   uint64_t& end) {
  const uint64_t chunk = (n + G - 1) / G;
  beg = (uint64_t)b * chunk;
  if (beg > n) beg = n;
  end = beg + chunk;
  if (end > n) end = n;
}

__global__ __launch_bounds__(BLOCK) void k_attr_count(int semantics, NodeArrays nodes,
                                                      uint64_t n_nodes, const uint64_t* mbase,
                                                      uint32_t n_meshes, uint32_t G,
                                                      uint64_t* partial) {
  if (nodes.skip && *nodes.skip) return;  // graph replay over changed sizes
  __shared__ uint64_t tmp[4];
  uint64_t beg, end;
  block_range(n_nodes, G, blockIdx.x, beg, end);
  uint64_t sv = 0, se = 0, sf = 0;
  AttrOut none = {nullptr, nullptr, nullptr, nullptr};
  uint32_t m = beg < end ? find_mesh64(mbase, n_meshes, beg) : 0;
  for (uint64_t t = beg + threadIdx.x; t < end; t += BLOCK) {
    while (m + 1 < n_meshes && mbase[m + 1] <= t) ++m;
    const AttrCounts c = node_attrs<false>(semantics, nodes, t, t - mbase[m], 0, 0, 0, none);
    sv += c.v;
    se += c.e;
    sf += c.f;
  }
  uint64_t tv, te, tf;
  block_excl_scan256(sv, tmp, tv);
  block_excl_scan256(se, tmp, te);
  block_excl_scan256(sf, tmp, tf);
  if (threadIdx.x == 0) {
    partial[3 * blockIdx.x] = tv;
    partial[3 * blockIdx.x + 1] = te;
    partial[3 * blockIdx.x + 2] = tf;
  }
}

__global__ __launch_bounds__(BLOCK) void k_triple_scan(uint64_t* partial, uint32_t G,
                                                       unsigned long long* totals) {
  __shared__ uint64_t tmp[4];
  const uint32_t per = (G + BLOCK - 1) / BLOCK;
  const uint32_t b0 = threadIdx.x * per;
  for (int c = 0; c < 3; ++c) {
    uint64_t s = 0;
    for (uint32_t k = 0; k < per; ++k)
      if (b0 + k < G) s += partial[3 * (b0 + k) + c];
    uint64_t tot;
    uint64_t run = block_excl_scan256(s, tmp, tot);
    for (uint32_t k = 0; k < per; ++k)
      if (b0 + k < G) {
        const uint64_t v = partial[3 * (b0 + k) + c];
        partial[3 * (b0 + k) + c] = run;
        run += v;
      }
    if (threadIdx.x == 0) totals[c] = tot;
  }
}

__global__ __launch_bounds__(BLOCK) void k_attr_write(int semantics, NodeArrays nodes,
                                                      uint64_t n_nodes, const uint64_t* mbase,
                                                      uint32_t n_meshes, uint32_t G,
                                                      const uint64_t* partial, AttrOut out,
                                                      uint64_t* mesh_first) {
  if (nodes.skip && *nodes.skip) return;  // graph replay over changed sizes
  __shared__ uint64_t tmp[4];
  uint64_t beg, end;
  block_range(n_nodes, G, blockIdx.x, beg, end);
  uint64_t bv = partial[3 * blockIdx.x], be = partial[3 * blockIdx.x + 1],
           bf = partial[3 * blockIdx.x + 2];
  AttrOut none = {nullptr, nullptr, nullptr, nullptr};
  uint32_t m = beg < end ? find_mesh64(mbase, n_meshes, beg) : 0;
  for (uint64_t tb = beg; tb < end; tb += BLOCK) {
    const uint64_t t = tb + threadIdx.x;
    AttrCounts c = {0, 0, 0};
    uint64_t local = 0;
    if (t < end) {
      while (m + 1 < n_meshes && mbase[m + 1] <= t) ++m;
      local = t - mbase[m];
      c = node_attrs<false>(semantics, nodes, t, local, 0, 0, 0, none);
    }
    uint64_t tv, te, tf;
    const uint64_t ov = block_excl_scan256((uint64_t)c.v, tmp, tv) + bv;
    const uint64_t oe = block_excl_scan256((uint64_t)c.e, tmp, te) + be;
    const uint64_t of = block_excl_scan256((uint64_t)c.f, tmp, tf) + bf;
    if (t < end) {
      node_attrs<true>(semantics, nodes, t, local, ov, oe, of, out);
      if (local == 0) {
        mesh_first[3 * m] = ov;
        mesh_first[3 * m + 1] = oe;
        mesh_first[3 * m + 2] = of;
      }
    }
    bv += tv;
    be += te;
    bf += tf;
  }
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

void launch_fill_u32(uint32_t* p, uint32_t value, uint64_t n, hipStream_t s) {
  if (n == 0) return;
  const uint64_t blocks = std::min<uint64_t>(grid_for((n + 3) / 4), 1u << 20);
  hipLaunchKernelGGL(k_fill_u32, dim3((uint32_t)blocks), dim3(BLOCK), 0, s, p, value, n);
}

template <typename K>
void launch_neighbors_level(int level, KeyLayout<K> kl, const void* elem_next,
                            const uint32_t* elem_group_next, uint64_t n_groups,
                            const LevelSpan* spans, uint32_t n_levels,
                            const MeshTreeState* state, const MeshNodeLayout* layout,
                            NodeArrays nodes, hipStream_t s) {
  if (n_groups == 0) return;
  hipLaunchKernelGGL(k_neighbors_level<K>, dim3(grid_for(8 * n_groups)), dim3(BLOCK), 0, s,
                     level, kl, (const K*)elem_next, elem_group_next, n_groups, spans, n_levels,
                     state, layout, nodes);
}

size_t attr_tmp_bytes(uint32_t blocks) { return (size_t)3 * blocks * sizeof(uint64_t); }

void launch_attrs_count(int semantics, const NodeArrays& nodes, uint64_t n_nodes,
                        const uint64_t* mesh_node_base, uint32_t n_meshes, uint32_t blocks,
                        void* tmp, AttrOut out, hipStream_t s) {
  uint64_t* partial = (uint64_t*)tmp;
  hipLaunchKernelGGL(k_attr_count, dim3(blocks), dim3(BLOCK), 0, s, semantics, nodes, n_nodes,
                     mesh_node_base, n_meshes, blocks, partial);
  hipLaunchKernelGGL(k_triple_scan, dim3(1), dim3(BLOCK), 0, s, partial, blocks, out.totals);
}

void launch_attrs_write(int semantics, const NodeArrays& nodes, uint64_t n_nodes,
                        const uint64_t* mesh_node_base, uint32_t n_meshes, uint32_t blocks,
                        void* tmp, AttrOut out, hipStream_t s) {
  uint64_t* partial = (uint64_t*)tmp;
  uint64_t* mesh_first = (uint64_t*)out.totals + 4;  // [3 * n_meshes] after the totals
  hipLaunchKernelGGL(k_attr_write, dim3(blocks), dim3(BLOCK), 0, s, semantics, nodes, n_nodes,
                     mesh_node_base, n_meshes, blocks, (const uint64_t*)partial, out, mesh_first);
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

#define SVO_INST(K)                                                                              \
  template void launch_emit<K>(const EmitArgs<K>&, hipStream_t);                                 \
  template void launch_neighbors_level<K>(int, KeyLayout<K>, const void*, const uint32_t*,       \
                                          uint64_t, const LevelSpan*, uint32_t,                  \
                                          const MeshTreeState*, const MeshNodeLayout*,           \
                                          NodeArrays, hipStream_t);
SVO_INST(uint32_t)
SVO_INST(uint64_t)
#undef SVO_INST

}  // namespace svo
