// svo_internal.h -- host-side declarations shared by the pipeline and the
// kernel translation units.  Every launcher takes device pointers and a
// stream and enqueues work only; none of them synchronises.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "svo_device.h"

namespace svo {

// ------------------------------------------------------------ tuning knobs
constexpr int SIZE_CLASSES = 15;

struct Tuning {
  uint32_t small_max_cells = 1024;  // largest box (cells) whose triangle shares a wave
  uint32_t sort_blocks = 65536;     // grid bound of the radix sort passes (tiles stride)
  uint32_t scan_blocks = 1024;      // fixed grid of the level / attribute scans
  // Occupancy bitmap instead of the sort (level 1 straight from the bitmap)
  // while the bitmap is at most this many bytes and at most this many bytes
  // per candidate cell (so sparse hits in a huge grid still take the sort).
  uint64_t bitmap_max_bytes = 32ull << 30;
  uint32_t bitmap_bytes_per_cell = 64;
  int force_path = 0;               // 0 automatic, 1 bitmap, 2 sort
  // svo_build_batch runs batches of at least 2 * batch_min_meshes meshes as
  // up to batch_lanes concurrent passes
  uint32_t batch_lanes = 2;
  uint32_t batch_min_meshes = 16;
  // The same per size class (size_class_of); 0 = small_max_cells.  Set by the tuning search.
  uint32_t class_small_max[SIZE_CLASSES] = {};
};

// Size class of a mesh for tuning: 5 resolution bands (max axis <= 64, 128,
// 256, 512, above) x 3 bands of res^2 / triangles, which grows with the
// triangles' edge length in voxels for a surface spanning its box (<= 4:
// triangles of about a voxel or less, <= 64: a few voxels, above: larger).
inline int size_class_of(const int32_t res[3], uint64_t n_tris) {
  const int32_t r = res[0] > res[1] ? (res[0] > res[2] ? res[0] : res[2])
                                    : (res[1] > res[2] ? res[1] : res[2]);
  const int band = r <= 64 ? 0 : r <= 128 ? 1 : r <= 256 ? 2 : r <= 512 ? 3 : 4;
  const double q = (double)r * (double)r / (double)(n_tris ? n_tris : 1);
  const int qb = q <= 4.0 ? 0 : q <= 64.0 ? 1 : 2;
  return 3 * band + qb;
}

// ------------------------------------------------------------ k_voxelize.hip
// What a pass sets up before its first kernel, in one launch: `n_table` words
// copied from pinned host memory (0: they are in place), the boxes `acc` (8
// words a mesh) at their start values, `n_zero` words cleared.
struct PassBegin {
  const uint32_t* host_table;
  uint32_t* table;
  uint64_t n_table;
  uint32_t* acc;
  uint32_t n_meshes;
  uint32_t* zero;
  uint64_t n_zero;
};
void launch_begin(const PassBegin& B, hipStream_t s);
// Per-mesh ordered-float min/max of all points, and whether a coordinate is
// not finite or an index out of range (8 x uint32 per mesh, launch_begin's acc).
void launch_bbox(const MeshDev* meshes, uint32_t n_meshes, uint64_t max_points, uint64_t max_tris,
                 uint32_t* acc, hipStream_t s);
// A pass's counters: COUNT_SLOTS slots of a cache line each, since atomics on
// one address serialize; a total is the sum over the slots.
constexpr uint32_t COUNT_SLOTS = 64, COUNT_STRIDE = 8;
constexpr uint32_t COUNT_HITS = 0, COUNT_CELLS = 1, COUNT_CHUNKS = 2;
// Grid parameters from the boxes (BaseModel.h:24-73, SVO.cu:342-351); candidate
// cells and big-triangle chunk counts, added to `slots`.
void launch_classify(const MeshDev* meshes, const uint32_t* acc, MeshParams* params,
                     const uint64_t* tri_base, uint32_t n_meshes, uint64_t n_tris,
                     const Tuning& tn, unsigned long long* slots, hipStream_t s);
// Candidate cells and chunks to out[0], out[1] (device or pinned host memory).
void launch_read_totals(const unsigned long long* slots, unsigned long long* out, hipStream_t s);
// Surface voxelization (SVO.cu:37-188): emits composite keys.
// Hits go to `keys` (raw, for the sort; *key_count receives their number) when
// `bitmap` is null, else into the occupancy bitmap (word bm_off[mesh] + code /
// 32, bit code % 32, which the caller has zeroed; counted in `slots`).  With
// `line_flags`, byte k of it (zeroed as well) is set for each line of
// BITMAP_LINE_BYTES bitmap bytes that receives a bit.
constexpr uint64_t BITMAP_LINE_BYTES = 64;
template <typename K>
void launch_voxelize(const MeshDev* meshes, const MeshParams* params, const uint64_t* tri_base,
                     uint32_t n_meshes, uint64_t n_tris, int cb, const Tuning& tn, K* keys,
                     uint32_t* bitmap, const uint64_t* bm_off, uint8_t* line_flags,
                     unsigned long long* key_count, unsigned long long* slots, BigItem* big,
                     unsigned long long* big_count, uint64_t big_cap, hipStream_t s);

// ------------------------------------------------------------ k_sort.hip
// LSD radix sort of n (device-resident count) keys on bits [0, bits).
// Returns in *result which of (a, b) holds the sorted keys; a null result asks
// for them in a.  n must not exceed cap; `tmp` needs radix_sort_tmp_bytes(cap)
// bytes.  `blocks` bounds the persistent grid of the digit passes.
size_t radix_sort_tmp_bytes(uint64_t cap);
size_t radix_sort_tmp_bound(uint64_t cap);  // over all capacities up to cap
template <typename K>
void launch_radix_sort(K* a, K* b, const unsigned long long* n, uint64_t cap, int bits,
                       uint32_t blocks, void* tmp, K** result, hipStream_t s);

// ------------------------------------------------------------ k_levels.hip
struct LevelArrays {
  void* elem;            // K[cap]: sorted unique keys of this level (S_l)
  uint32_t* elem_group;  // [cap]: group index (at this level) of each element (l >= 2)
  uint32_t* first_child; // [cap]: for groups of the level below: first member index
  uint8_t* kids;         // [cap]: for groups of the level below: bit k set if child 8p + k exists
  uint64_t cap;
};
// Level 1 from the sorted hit keys: unique codes, their groups, and the
// level-2 element array (parents).  Counts go to counts[0] (level 1 elements)
// and counts[1] (level 2 elements).  n_sorted <= cap; `blocks` bounds the
// persistent grid; `tmp` needs level_tmp_bytes(cap) bytes and is shared with
// the later levels of the same pass (launch_level_first prepares it).  l2.kids
// may be null (no child masks).
template <typename K>
void launch_level_first(const K* sorted, const unsigned long long* n_sorted, uint64_t cap,
                        KeyLayout<K> kl, LevelArrays l1, LevelArrays l2,
                        unsigned long long* counts, LevelSpan* spans1, uint32_t n_levels,
                        uint32_t blocks, void* tmp, hipStream_t s);
// Level 1 from the occupancy bitmap (n_words words; mesh m owns words
// [bm_off[m], bm_off[m+1]), and every bm_off[m] is a multiple of
// BITMAP_TILE_WORDS): the same outputs as launch_level_first followed
// by launch_level_first_finalize, and the bitmap is left all zero (the bytes
// that takes are added to *reset_bytes); totals[0..2] receive the counters'
// sums (candidate cells, chunks, raw hits).  With the flags of launch_voxelize (one
// mesh, bm_off[0] = 0) only the flagged lines are read; `line_list` receives
// their numbers.  `tmp` needs
// bitmap_level_tmp_bytes(n_words); `lvl_tmp` (level_tmp_bytes of l1.cap) is
// prepared for the later levels.
size_t bitmap_level_tmp_bytes(uint64_t n_words);
// Words per tile of the bitmap's level-1 pass; each mesh's bitmap region
// starts on a tile boundary, so that no tile holds two meshes' words.
constexpr uint64_t BITMAP_TILE_WORDS = 2048;
inline uint64_t bitmap_region_words(uint64_t codes) {
  return ((codes + 31) / 32 + BITMAP_TILE_WORDS - 1) / BITMAP_TILE_WORDS * BITMAP_TILE_WORDS;
}
template <typename K>
void launch_level_first_bitmap(uint32_t* bits, uint64_t n_words, const uint64_t* bm_off,
                               uint32_t n_meshes, KeyLayout<K> kl, LevelArrays l1,
                               LevelArrays l2, unsigned long long* counts, LevelSpan* spans1,
                               uint32_t n_levels, MeshTreeState* state, void* tmp,
                               void* lvl_tmp, unsigned long long* reset_bytes,
                               const unsigned long long* slots, unsigned long long* totals,
                               const uint8_t* line_flags, uint32_t* line_list, hipStream_t s);
// Marks meshes whose level-1 set holds a single voxel as depth-1 trees (the
// sort path; launch_level_first_bitmap does it itself).
void launch_level_first_finalize(const LevelSpan* spans, uint32_t n_meshes, uint32_t n_levels,
                                 MeshTreeState* state, hipStream_t s);
// Levels 2 .. n_levels (at most 23; level l's arrays at lv[l], up to n_levels +
// 1): roots of meshes whose level holds one element; groups of the others feed
// the next level.
template <typename K>
void launch_levels(KeyLayout<K> kl, const LevelArrays* lv, uint32_t n_levels,
                   unsigned long long* counts, LevelSpan* spans, MeshTreeState* state,
                   uint32_t blocks, void* tmp, hipStream_t s);
size_t level_tmp_bytes(uint64_t cap);

// ------------------------------------------------------------ k_attrs.hip
// Per mesh node layout computed on the host after the level phase.
struct MeshNodeLayout {
  uint64_t node_base;    // first node of the mesh in the batch arrays
  uint64_t n_nodes;
  uint32_t depth;
  uint64_t level_off[24];// node offset of each level within the mesh (level l at [l-1])
  float width[24];       // node width per level
};

// A run of consecutive nodes of one mesh and level, or one root, in node
// order; computed on the host beside the layout.  Node t of a level's run is
// child (t - t0) & 7 of the level's parent group (t - t0) / 8.  One aligned
// record holds all that the emission needs of a run, so that a workgroup
// fetches it with one round of scalar loads.
struct alignas(64) NodeSeg {
  uint32_t t0, t1;   // nodes [t0, t1) of the pass
  uint32_t local0;   // index of node t0 within its mesh
  uint32_t level_kind;  // level in bits 0-7, SEG_* above
  uint32_t child0;   // children of the node whose first child is element i start at child0 + 8i
  uint32_t parent0;  // parent of group g: parent0 + 8 * elem_group[g] + (key & 7)
  float width;
  float origin[3];   // gridOrigin
  uint32_t mesh;
  uint32_t pad;
  // the run's parent groups (level + 1's arrays, from its first group on):
  // keys, their own groups, first children and child masks; a root's own key
  const void* elem;
  const uint32_t* group;
  const uint32_t* first_child;
  const uint8_t* kids;
};
enum : uint32_t {
  SEG_ROOT = 1u << 8,       // the root: child0 is its first child (level >= 2)
  SEG_ROOT_CHILD = 1u << 9, // children of the root: parent0 is the root
};

struct NodeArrays {
  void* code;            // uint32 or uint64 per node (code_bytes)
  uint8_t* is_leaf;
  float* origin;         // 3 per node
  float* width;
  uint32_t* parent;
  uint32_t* childs;      // 8 per node
  uint32_t* neighbors;   // 27 per node
  int code_bytes;
  // Graph-captured passes: when *skip is nonzero (a size differs from the
  // recorded run) the node, neighbor and record kernels return at once, so
  // that nothing is written past the recorded layout.  Null otherwise.
  const uint32_t* skip;
};

// Everything of a pass's output in one launch, in output order: node arrays,
// voxel codes and, as `neighbors` / `records` ask, the reference's neighbor
// slots and its vertex and edge records at the identity offsets (8 and 12
// per node, valid when no record can equal its predecessor).  Every output
// array starts on a 16-byte boundary and may be written up to the next one.
template <typename K>
struct EmitArgs {
  KeyLayout<K> kl;
  const NodeSeg* segs;        // in node order
  const uint32_t* seg_first;  // first node of each
  uint32_t n_segs, n_roots;
  uint64_t n_nodes;           // below 2^32 (more would not fit the device)
  NodeArrays out;
  const K* voxels_in;  // level-1 keys
  uint64_t n_voxels;
  void* voxels;
  svo_vertex_t* verts;
  svo_edge_t* edges;
  bool neighbors, records;
};
template <typename K>
void launch_emit(const EmitArgs<K>& a, hipStream_t s);
void launch_fill_u32(uint32_t* p, uint32_t value, uint64_t n, hipStream_t s);
// Copies `bytes` device bytes into a pinned ring of RING_SLOTS pieces from
// slot `slot` on (at most the whole ring), piece after piece; the RING_BLOCKS
// flags of a piece's slot become `number` when it has arrived.  Returns the
// launch's own status (hipGetLastError could be an earlier error of the thread).
constexpr size_t RING_PIECE = 512 << 10, RING_SLOTS = 16;
constexpr uint32_t RING_BLOCKS = 32;
hipError_t launch_ring_copy(const void* src, uint64_t bytes, void* ring, uint32_t* flags,
                            uint64_t slot, uint32_t number, hipStream_t s);
// Copies n words; either side may be pinned host memory.  For a pass's tables
// and readbacks of a few KB: 2 to 4 us, and less host time than asynchronous
// copies (five of them read the levels back in 25 to 40 us).
void launch_copy_u32(uint32_t* dst, const uint32_t* src, uint64_t n, hipStream_t s);
// Sets *flag (atomic OR of 1) when the `bytes` bytes (a multiple of 4, both
// 4-byte aligned) at `got` differ from those at `want`.
void launch_check_equal(const void* got, const void* want, uint64_t bytes, uint32_t* flag,
                        hipStream_t s);
// Neighbor rows of one level, intended semantics, from the rows of the level
// above, and (when `keep` is set) which records each node keeps.  The level's
// segments segs[level_segs[i]] own workgroups from level_blocks[i] on,
// neighbor_blocks(segment) each; the roots, whose rows need no level above,
// may stand among them.
uint32_t neighbor_blocks(const NodeSeg& seg);
void launch_neighbors_level(const NodeSeg* segs, const uint32_t* level_segs,
                            const uint32_t* level_blocks, uint32_t n_level_segs, uint32_t blocks,
                            int key_bytes, NodeArrays nodes, uint32_t* keep, hipStream_t s);
// Vertex, edge and face records by keep masks.
struct AttrOut {
  svo_vertex_t* verts;
  svo_edge_t* edges;
  svo_edge_t* faces;
  unsigned long long* totals;  // [3] totals, then from [4] on 3 first records per mesh
};
// `tmp` holds keep_bytes(n_nodes) bytes and begins with the nodes' keep masks
// (written by launch_neighbors_level; by this call, reference semantics).
size_t keep_bytes(uint64_t n_nodes);
template <typename K>
void launch_kept_records(int semantics, KeyLayout<K> kl, const NodeArrays& nodes, uint64_t n_nodes,
                         const NodeSeg* segs, const uint32_t* seg_first, uint32_t n_segs,
                         void* tmp, AttrOut out, hipStream_t s);
// The reference's vertex and edge records of given nodes (origin 3 floats and
// width 1 float each) at the identity offsets, owner = the node's index.
void launch_ref_records(const float* origin, const float* width, uint64_t n_nodes,
                        svo_vertex_t* verts, svo_edge_t* edges, hipStream_t s);
// 168-byte SVONode records for nodes [first, first + n) (32-bit codes).
void launch_pack_aos(const NodeArrays& nodes, uint64_t first, uint64_t n, void* dst,
                     hipStream_t s);
// The same with node, slot and out in pinned host memory; the first
// query_ring_blocks(n) flags become `number` when the answers are there.
// Returns the launch's own status.
uint32_t query_ring_blocks(uint64_t n);
hipError_t launch_query_ring(const uint32_t* neighbors, uint64_t n_nodes, const uint32_t* node,
                             const uint8_t* slot, uint64_t n, uint32_t* out, uint32_t* flags,
                             uint32_t number, hipStream_t s);
void launch_query_neighbors(const uint32_t* neighbors, uint64_t n_nodes, const uint32_t* node,
                            const uint8_t* slot, uint64_t n, uint32_t* out, hipStream_t s);

}  // namespace svo
