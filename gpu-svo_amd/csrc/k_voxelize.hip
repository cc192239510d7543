// k_voxelize.hip -- point bbox, grid parameters and surface voxelization.
//
// Follows the reference's surfaceVoxelize (SVO.cu:37-188): per triangle a
// plane test and three 2-D projection tests over every cell of the clamped
// bounding box, with the same float operation order (built with
// -ffp-contract=off, correctly rounded divide and sqrt, denormals kept).
//
// Work distribution (the reference gives one thread per triangle):
//  * k_classify   one lane per triangle: box cells -> key capacity and the
//                 number of big-triangle chunks (exact, read back once).
//  * k_vox_rows   one wave per run of triangles: a lane sets up a triangle,
//                 then the wave's lanes take the box rows (y, z) of all of
//                 them in turn.  Triangles over the size limit are queued in
//                 items of 512 rows, each a wave's work in a second launch.
// A row's cells are found from the x-interval that the tests leave, in place
// of testing each cell (below); the cells that rounding could decide either
// way are tested with the reference's float operations.
#include <algorithm>

#include "svo_internal.h"
#include "svo_scan.h"

namespace svo {
namespace {

constexpr int BLOCK = 256;
constexpr int WAVES = BLOCK / 64;
constexpr int STAGE = 1024;        // keys staged per wave

__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ inline uint64_t bcast_first(uint64_t v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return ((uint64_t)hi << 32) | lo;
}

__device__ inline uint32_t find_mesh(const uint64_t* base, uint32_t n_meshes, uint64_t gid) {
  uint32_t lo = 0, hi = n_meshes;  // base[lo] <= gid < base[hi]
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (base[mid] <= gid) lo = mid; else hi = mid;
  }
  return lo;
}

// The mesh of triangle gid >= first, `first` the same in every lane of the
// wave: one step of 64 comparisons per factor 64 of meshes finds the mesh of
// `first`, which nearly always is that of the whole wave.
__device__ inline uint32_t find_mesh_wave(const uint64_t* base, uint32_t n_meshes, uint64_t first,
                                          uint64_t gid) {
  uint32_t lo = 0, n = n_meshes;
  while (n > 1) {
    const uint32_t step = (n + 63) / 64, i = __lane_id() * step;
    const uint64_t at = __ballot(i < n && base[lo + i] <= first);
    const uint32_t last = 63u - (uint32_t)__builtin_clzll(at);  // base[lo] <= first
    lo += last * step;
    n = n - last * step < step ? n - last * step : step;
  }
  while (lo + 1 < n_meshes && base[lo + 1] <= gid) ++lo;
  return lo;
}

// ------------------------------------------------------------------ bbox
// Everything a pass sets up before its first kernel: the control tables from
// pinned host memory, the boxes at their start values, zeros.
__global__ __launch_bounds__(BLOCK) void k_begin(PassBegin B) {
  const uint64_t stride = (uint64_t)gridDim.x * BLOCK;
  const uint64_t i0 = (uint64_t)blockIdx.x * BLOCK + threadIdx.x;
  for (uint64_t i = i0; i < B.n_table; i += stride) B.table[i] = B.host_table[i];
  for (uint64_t i = i0; i < 8ull * B.n_meshes; i += stride)
    B.acc[i] = (i & 7) < 3 ? 0xFFFFFFFFu : 0u;  // ordered min starts at +max, max at 0
  for (uint64_t i = i0; i < B.n_zero; i += stride) B.zero[i] = 0u;
}

// Bounding boxes of the points (workgroups x < point_blocks) and a check of
// the triangles' indices (the others); acc[8 m ..]: ordered minima, maxima, a
// flag for a non-finite coordinate and one for an index out of range.  A
// workgroup takes its points and indices as dwords, twelve loads a thread in
// flight: 6.5 us for 163,842 points and 327,680 triangles (points taken one
// after the other in 41 workgroups and the indices in a launch of their own:
// 10.6 and 3).
constexpr int FLAT = 12;
constexpr uint32_t FLAT_CHUNK = BLOCK * FLAT;
constexpr uint32_t BBOX_BLOCKS = 256;  // per mesh: its six atomics follow each other
__global__ __launch_bounds__(BLOCK) void k_bbox(const MeshDev* meshes, uint32_t point_blocks,
                                                uint32_t* acc) {
  const MeshDev& md = meshes[blockIdx.y];
  uint32_t* a = acc + 8 * blockIdx.y;
  if (blockIdx.x >= point_blocks) {
    const uint64_t n = 3 * md.n_tris;
    const uint64_t n_points = md.n_points;
    uint32_t bad = 0;
    for (uint64_t start = (uint64_t)(blockIdx.x - point_blocks) * FLAT_CHUNK; start < n;
         start += (uint64_t)(gridDim.x - point_blocks) * FLAT_CHUNK) {
      int32_t v[FLAT];
#pragma unroll
      for (int j = 0; j < FLAT; ++j) {
        const uint64_t i = start + (uint64_t)j * BLOCK + threadIdx.x;
        v[j] = i < n ? md.tri[i] : 0;
      }
#pragma unroll
      for (int j = 0; j < FLAT; ++j) bad |= v[j] < 0 || (uint64_t)v[j] >= n_points;
    }
    if (__any(bad) && (threadIdx.x & 63) == 0) atomicOr(a + 7, 1u);
    return;
  }
  const uint64_t n = 3 * md.n_points;
  if ((uint64_t)blockIdx.x * FLAT_CHUNK >= n) return;
  // a thread's dword j is of axis (threadIdx.x + j) mod 3: FLAT_CHUNK and
  // BLOCK - 1 are multiples of 3
  static_assert(FLAT_CHUNK % 3 == 0 && BLOCK % 3 == 1 && FLAT % 3 == 0, "axes by position");
  uint32_t mn[3] = {0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu}, mx[3] = {0, 0, 0};
  uint32_t bad = 0;
  for (uint64_t start = (uint64_t)blockIdx.x * FLAT_CHUNK; start < n;
       start += (uint64_t)point_blocks * FLAT_CHUNK) {
    float v[FLAT];
#pragma unroll
    for (int j = 0; j < FLAT; ++j) {
      const uint64_t i = start + (uint64_t)j * BLOCK + threadIdx.x;
      v[j] = i < n ? md.pts[i] : md.pts[(threadIdx.x + j) % 3];  // the first point again
    }
#pragma unroll
    for (int j = 0; j < FLAT; ++j) {
      if (!isfinite(v[j])) {
        bad = 1;
        continue;
      }
      const uint32_t k = float_to_ordered(v[j]);
      mn[j % 3] = k < mn[j % 3] ? k : mn[j % 3];
      mx[j % 3] = k > mx[j % 3] ? k : mx[j % 3];
    }
  }
  // by axis: axis x is at (x - threadIdx.x) mod 3
  {
    const uint32_t r = threadIdx.x % 3;
    const uint32_t n0 = mn[0], n1 = mn[1], n2 = mn[2], x0 = mx[0], x1 = mx[1], x2 = mx[2];
    mn[0] = r == 0 ? n0 : r == 1 ? n2 : n1;
    mn[1] = r == 0 ? n1 : r == 1 ? n0 : n2;
    mn[2] = r == 0 ? n2 : r == 1 ? n1 : n0;
    mx[0] = r == 0 ? x0 : r == 1 ? x2 : x1;
    mx[1] = r == 0 ? x1 : r == 1 ? x0 : x2;
    mx[2] = r == 0 ? x2 : r == 1 ? x1 : x0;
  }
  for (int off = 32; off > 0; off >>= 1) {
    for (int x = 0; x < 3; ++x) {
      const uint32_t omn = __shfl_xor(mn[x], off);
      const uint32_t omx = __shfl_xor(mx[x], off);
      mn[x] = omn < mn[x] ? omn : mn[x];
      mx[x] = omx > mx[x] ? omx : mx[x];
    }
    bad |= __shfl_xor(bad, off);
  }
  __shared__ uint32_t red[WAVES][7];
  const uint32_t w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    for (int x = 0; x < 3; ++x) {
      red[w][x] = mn[x];
      red[w][3 + x] = mx[x];
    }
    red[w][6] = bad;
  }
  __syncthreads();
  if (threadIdx.x < 7) {
    uint32_t v = red[0][threadIdx.x];
    for (int k = 1; k < WAVES; ++k) {
      const uint32_t o = red[k][threadIdx.x];
      if (threadIdx.x < 3) v = o < v ? o : v;
      else if (threadIdx.x < 6) v = o > v ? o : v;
      else v |= o;
    }
    if (threadIdx.x < 3) atomicMin(a + threadIdx.x, v);
    else if (threadIdx.x < 6) atomicMax(a + threadIdx.x, v);
    else if (v) atomicOr(a + 6, 1u);
  }
}

// createMeshBBCube (BaseModel.h:24-49) and the voxel size (SVO.cu:348-350).
__device__ inline MeshParams mesh_params(const MeshDev& md, const uint32_t* a) {
  MeshParams P;
  P.status = (a[6] ? ERR_NONFINITE : 0u) | (a[7] ? ERR_INDEX : 0u);
  float mn[3], mx[3], len[3], amin[3], amax[3];
  for (int k = 0; k < 3; ++k) {
    mn[k] = ordered_to_float(a[k]);
    mx[k] = ordered_to_float(a[3 + k]);
    len[k] = mx[k] - mn[k];
    amin[k] = mn[k];
    amax[k] = mx[k];
    P.res[k] = md.res[k];
  }
  const float max_length = fmax_r(len[0], fmax_r(len[1], len[2]));
  if (!(max_length > 0.0f)) P.status |= ERR_DEGENERATE;
  for (int k = 0; k < 3; ++k) {
    if (max_length == len[k]) continue;
    const float delta = max_length - len[k];
    amin[k] = mn[k] - (delta / 2.0f);
    amax[k] = mx[k] + (delta / 2.0f);
  }
  for (int k = 0; k < 3; ++k) {
    const float eps = (amax[k] - amin[k]) / 10001.0f;
    amin[k] -= eps;
    amax[k] += eps;
  }
  for (int k = 0; k < 3; ++k) {
    P.bmin[k] = amin[k];
    P.bmax[k] = amax[k];
    P.width[k] = amax[k] - amin[k];
    P.origin[k] = amin[k];
    P.unit[k] = P.width[k] / (float)P.res[k];
  }
  return P;
}

// ------------------------------------------------------------------ triangle setup
struct TriSetup {
  float n[3];
  float d1, d2;
  float ne[3][3][2];  // [plane xy|yz|zx][edge][2]
  float de[3][3];
  float u[3];
  int g0[3], g1[3];
};

// Loads a triangle relative to gridOrigin (SVO.cu:58-63).  false on a bad index.
__device__ inline bool load_tri(const MeshDev& md, const MeshParams& P, uint64_t local,
                                float v[3][3]) {
  const int32_t* t = md.tri + 3 * local;
  for (int k = 0; k < 3; ++k) {
    const int32_t i = t[k];
    if (i < 0 || (uint64_t)i >= md.n_points) return false;
    for (int a = 0; a < 3; ++a) v[k][a] = md.pts[3 * (uint64_t)i + a] - P.origin[a];
  }
  return true;
}

// Triangle box in grid cells (SVO.cu:73-85).
__device__ inline void tri_box(const float v[3][3], const MeshParams& P, int g0[3], int g1[3]) {
  for (int a = 0; a < 3; ++a) {
    const float lo = fmin_r(v[0][a], fmin_r(v[1][a], v[2][a]));
    const float hi = fmax_r(v[0][a], fmax_r(v[1][a], v[2][a]));
    g0[a] = clamp_i((int)(lo / P.unit[a]), 0, P.res[a] - 1);
    g1[a] = clamp_i((int)(hi / P.unit[a]), 0, P.res[a] - 1);
  }
}

// Plane and projection test constants (SVO.cu:65-149).
__device__ inline void tri_setup(const float v[3][3], const MeshParams& P, TriSetup& S) {
  float e[3][3];
  for (int a = 0; a < 3; ++a) {
    e[0][a] = v[1][a] - v[0][a];
    e[1][a] = v[2][a] - v[1][a];
    e[2][a] = v[0][a] - v[2][a];
    S.u[a] = P.unit[a];
  }
  float n0 = e[0][1] * e[1][2] - e[0][2] * e[1][1];
  float n1 = e[0][2] * e[1][0] - e[0][0] * e[1][2];
  float n2 = e[0][0] * e[1][1] - e[0][1] * e[1][0];
  const float zz = n0 * n0 + (n1 * n1 + n2 * n2);  // squaredNorm, a0 + (a1 + a2)
  if (zz > 0.0f) {
    const float s = sqrtf(zz);
    n0 = n0 / s;
    n1 = n1 / s;
    n2 = n2 / s;
  }
  S.n[0] = n0;
  S.n[1] = n1;
  S.n[2] = n2;
  tri_box(v, P, S.g0, S.g1);
  const float c0 = n0 > 0.0f ? S.u[0] : 0.0f;
  const float c1 = n1 > 0.0f ? S.u[1] : 0.0f;
  const float c2 = n2 > 0.0f ? S.u[2] : 0.0f;
  S.d1 = n0 * (c0 - v[0][0]) + (n1 * (c1 - v[0][1]) + n2 * (c2 - v[0][2]));
  S.d2 = n0 * ((S.u[0] - c0) - v[0][0]) +
         (n1 * ((S.u[1] - c1) - v[0][1]) + n2 * ((S.u[2] - c2) - v[0][2]));
  const bool flip[3] = {n2 < 0.0f, n0 < 0.0f, n1 < 0.0f};
  // plane p uses axes (a, b): xy = (0, 1), yz = (1, 2), zx = (2, 0)
  for (int p = 0; p < 3; ++p) {
    const int a = p, b = (p + 1) % 3;
    for (int i = 0; i < 3; ++i) {
      float x0 = -1.0f * e[i][b];
      float x1 = e[i][a];
      if (flip[p]) {
        x0 = -x0;
        x1 = -x1;
      }
      S.ne[p][i][0] = x0;
      S.ne[p][i][1] = x1;
      S.de[p][i] = ((-1.0f * (x0 * v[i][a] + x1 * v[i][b])) + fmax_r(0.0f, S.u[a] * x0)) +
                   fmax_r(0.0f, S.u[b] * x1);
    }
  }
}

// Rows by interval.  In row (y, z) each of the seven tests left (plane, three
// xy edges, three zx edges) is affine in x, so that the cells that pass are
// those between the tests' roots.  A root is found in float as
// -(row terms) * (1 / slope) and is wrong, together with the rounding of the
// test itself, by less than
//   9 u M / |slope|,  M = |slope| * (largest x + 1) + |row terms|,  u = 2^-24,
// slope per cell and M over the triangle's box: the test (two products, two
// sums) rounds within 4 u M; the sum of the row terms, the slope, its
// reciprocal and the root within 4 u M / |slope|; the root +- e within
// u M / |slope|.  e = 12 u M / |slope| leaves a third for the rounding of M
// and e themselves.  So a cell beyond root +- e fails for certain, one inside
// root -+ e passes for certain, and the few between are tested as the
// reference does (cell_hit).  A test of slope zero bounds nothing (error
// ROW_FREE: no cell is certain).  Where a test's M is so small or large that
// its products could underflow or overflow, or is no number, every cell of the
// triangle's box goes to cell_hit.
constexpr float ROW_ERR = 12.0f * 0x1p-24f, ROW_FREE = 1e30f;

// What a row needs of its triangle, in 15 16-byte pieces of LDS.
struct alignas(16) RowTri {
  float yz[3][4];                // ne.y, ne.z, de of the yz edges; n.y, n.z, u.y
  float uz, inv_ny; int32_t y0, z0;
  float xy_y[3], nx;             // y slopes of the xy edges
  float zx_z[3], d1;             // z slopes of the zx edges
  float xy_d[3], d2;
  float zx_d[3], ux;
  float inv[7]; int32_t ny;      // 1 / slope: plane, xy edges, zx edges
  float err[7]; int32_t x0;      // e of the same
  float xy_x[3]; int32_t x1;     // x slopes (cell_hit only)
  float zx_x[3]; uint32_t row0;  // item index - row
  uint32_t key_lo, key_hi;       // mesh key or first 64-bit bitmap word
  uint32_t exact, pad;           // nonzero: no interval holds
};
static_assert(sizeof(RowTri) == 15 * 16, "fifteen pieces");

// False when M lies outside (lo, hi) (also for NaN).
__device__ inline bool row_bound(float slope, float rest, float xmax, float lo, float hi,
                                 float& inv, float& err) {
  const float b = fabsf(slope), M = b * xmax + rest;
  inv = 1.0f / slope;
  err = M * fabsf(inv) * ROW_ERR;
  if (!(b > 0.0f && err < ROW_FREE)) {
    inv = 0.0f;
    err = ROW_FREE;
  }
  return M > lo && M < hi;
}

__device__ inline void row_setup(const TriSetup& S, RowTri& T) {
  bool ok = true;
  const float xmax = (float)S.g1[0] + 1.0f, ymax = ((float)S.g1[1] + 1.0f) * S.u[1],
              zmax = ((float)S.g1[2] + 1.0f) * S.u[2];
  for (int i = 0; i < 3; ++i) {
    T.yz[i][0] = S.ne[1][i][0];
    T.yz[i][1] = S.ne[1][i][1];
    T.yz[i][2] = S.de[1][i];
    T.xy_x[i] = S.ne[0][i][0];
    T.xy_y[i] = S.ne[0][i][1];
    T.zx_z[i] = S.ne[2][i][0];
    T.zx_x[i] = S.ne[2][i][1];
    T.xy_d[i] = S.de[0][i];
    T.zx_d[i] = S.de[2][i];
    ok &= row_bound(S.ne[0][i][0] * S.u[0], fabsf(S.ne[0][i][1]) * ymax + fabsf(S.de[0][i]),
                    xmax, 0x1p-90f, 0x1p100f, T.inv[1 + i], T.err[1 + i]);
    ok &= row_bound(S.ne[2][i][1] * S.u[0], fabsf(S.ne[2][i][0]) * zmax + fabsf(S.de[2][i]),
                    xmax, 0x1p-90f, 0x1p100f, T.inv[4 + i], T.err[4 + i]);
  }
  // the plane test multiplies two such values
  ok &= row_bound(S.n[0] * S.u[0],
                  fabsf(S.n[1]) * ymax + fabsf(S.n[2]) * zmax + fabsf(S.d1) + fabsf(S.d2), xmax,
                  0x1p-50f, 0x1p60f, T.inv[0], T.err[0]);
  T.exact = ok ? 0u : 1u;
  T.yz[0][3] = S.n[1];
  T.yz[1][3] = S.n[2];
  T.yz[2][3] = S.u[1];
  T.uz = S.u[2];
  T.nx = S.n[0];
  T.d1 = S.d1;
  T.d2 = S.d2;
  T.ux = S.u[0];
  T.x0 = S.g0[0];
  T.x1 = S.g1[0];
  T.y0 = S.g0[1];
  T.z0 = S.g0[2];
  T.ny = S.g1[1] - S.g0[1] + 1;
  T.inv_ny = 1.0f / (float)T.ny;
}

// The reference's terms of row (y, z): everything of the 13 tests that does
// not depend on x.  False when a yz-projection test fails (the row is empty).
struct RowTerms {
  float A;       // n.y*p.y + n.z*p.z  (inner sum of n.dot(p))
  float rxy[3];  // ne_xy[i].y * p.y
  float rzx[3];  // ne_zx[i].x * p.z
};
__device__ inline bool row_terms(const RowTri& T, int y, int z, RowTerms& R) {
  const float py = (float)y * T.yz[2][3];
  const float pz = (float)z * T.uz;
  bool ok = true;
  for (int i = 0; i < 3; ++i) ok &= !((T.yz[i][0] * py + T.yz[i][1] * pz) + T.yz[i][2] < 0.0f);
  R.A = T.yz[0][3] * py + T.yz[1][3] * pz;
  for (int i = 0; i < 3; ++i) {
    R.rxy[i] = T.xy_y[i] * py;
    R.rzx[i] = T.zx_z[i] * pz;
  }
  return ok;
}
// The reference's tests of cell x of the row.
__device__ inline bool cell_hit(const RowTri& T, const RowTerms& R, int x) {
  const float px = (float)x * T.ux;
  const float t = T.nx * px + R.A;
  bool ok = !((t + T.d1) * (t + T.d2) > 0.0f);
  for (int i = 0; i < 3; ++i) {
    ok &= !((T.xy_x[i] * px + R.rxy[i]) + T.xy_d[i] < 0.0f);
    ok &= !((R.rzx[i] + T.zx_x[i] * px) + T.zx_d[i] < 0.0f);
  }
  return ok;
}

// Cells [xa, xb] of the row may hit, [ia, ib] hit for certain (either may be
// empty).
__device__ inline void row_range(const RowTri& T, const RowTerms& R, int& xa, int& xb, int& ia,
                                 int& ib) {
  float lo = (float)T.x0, hi = (float)T.x1, ilo = lo, ihi = hi;
  {
    const float r1 = (-T.d1 - R.A) * T.inv[0], r2 = (-T.d2 - R.A) * T.inv[0];
    const float a = fminf(r1, r2), b = fmaxf(r1, r2), e = T.err[0];
    lo = fmaxf(lo, a - e);
    hi = fminf(hi, b + e);
    ilo = fmaxf(ilo, a + e);
    ihi = fminf(ihi, b - e);
  }
#pragma unroll
  for (int i = 1; i < 7; ++i) {
    const float c = i < 4 ? R.rxy[i - 1] + T.xy_d[i - 1] : R.rzx[i - 4] + T.zx_d[i - 4];
    const float inv = T.inv[i], e = T.err[i], root = -c * inv;
    // rising tests pass above their root, falling ones below; an unused test
    // (inv 0) counts as falling with root 0
    const bool up = inv > 0.0f;
    lo = fmaxf(lo, up ? root - e : -ROW_FREE);
    ilo = fmaxf(ilo, up ? root + e : -ROW_FREE);
    hi = fminf(hi, up ? ROW_FREE : root + e);
    ihi = fminf(ihi, up ? ROW_FREE : root - e);
  }
  const float below = (float)T.x0 - 1.0f, above = (float)T.x1 + 1.0f;
  xa = (int)ceilf(fminf(lo, above));
  xb = (int)floorf(fmaxf(hi, below));
  ia = (int)ceilf(fminf(ilo, above));
  ib = (int)floorf(fmaxf(ihi, below));
  if (T.exact) {
    xa = T.x0;
    xb = T.x1;
    ia = 0;
    ib = -1;
  }
}

// Where a voxelization kernel puts its hits: keys (staged, for the sort) or
// the occupancy bitmap.
template <typename K>
struct VoxOut {
  K* keys;                // key path
  uint32_t* bits;         // bitmap path
  const uint64_t* bm_off; // bitmap words before each mesh
  uint8_t* line_flags;    // bitmap path: a byte per 64-byte line, or null
  unsigned long long* count;  // key path: keys stored
  unsigned long long* slots;  // bitmap path: hits are counted in the slots
};

// Big-triangle work item: 512 rows (y, z) of the box.
constexpr uint64_t BIG_ROWS = 512;
constexpr uint64_t BIG_BLOCKS = 8192;

// The meshes' parameters from their boxes, and the candidate cells and
// big-triangle chunk counts, added to the pass's counter slots: an atomic per
// workgroup, which on one address follow each other at 14 ns (327,680
// triangles: 18 us that way, 9 with the slots).
constexpr uint32_t CLASSIFY_BLOCKS = 1024;
__global__ __launch_bounds__(BLOCK) void k_classify(const MeshDev* meshes, const uint32_t* acc,
                                                    MeshParams* params, const uint64_t* tri_base,
                                                    uint32_t n_meshes, uint64_t n_tris,
                                                    uint32_t small_max,
                                                    unsigned long long* slots) {
  uint64_t cells = 0, chunks = 0;
  const uint64_t stride = (uint64_t)gridDim.x * BLOCK;
  const uint64_t gid0 = (uint64_t)blockIdx.x * BLOCK + threadIdx.x;
  for (uint64_t m = gid0; m < n_meshes; m += stride)
    params[m] = mesh_params(meshes[m], acc + 8 * m);
  uint32_t last_m = 0xFFFFFFFFu;
  MeshParams P;
  for (uint64_t gid = gid0; gid < n_tris; gid += stride) {
    const uint32_t m = find_mesh(tri_base, n_meshes, gid);
    const MeshDev& md = meshes[m];
    if (m != last_m) {
      P = mesh_params(md, acc + 8ull * m);
      last_m = m;
    }
    float v[3][3];
    if (P.status == 0 && load_tri(md, P, gid - md.tri_base, v)) {
      int g0[3], g1[3];
      tri_box(v, P, g0, g1);
      const uint64_t nx = g1[0] - g0[0] + 1, ny = g1[1] - g0[1] + 1, nz = g1[2] - g0[2] + 1;
      const uint64_t c = nx * ny * nz;
      const uint64_t sm = md.small_max ? md.small_max : small_max;
      cells += c;
      if (c > sm) chunks += (ny * nz + BIG_ROWS - 1) / BIG_ROWS;
    }
  }
  for (int off = 32; off > 0; off >>= 1) {
    cells += __shfl_xor(cells, off);
    chunks += __shfl_xor(chunks, off);
  }
  __shared__ uint64_t red[WAVES][2];
  if ((threadIdx.x & 63) == 0) {
    red[threadIdx.x >> 6][0] = cells;
    red[threadIdx.x >> 6][1] = chunks;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    uint64_t t = 0;
    for (int w = 0; w < WAVES; ++w) t += red[w][threadIdx.x];
    unsigned long long* slot = slots + (blockIdx.x % COUNT_SLOTS) * COUNT_STRIDE;
    if (t) atomicAdd(slot + COUNT_CELLS + threadIdx.x, (unsigned long long)t);
  }
}

__global__ void k_read_totals(const unsigned long long* slots, unsigned long long* out) {
  const unsigned long long* slot = slots + threadIdx.x * COUNT_STRIDE;
  const uint64_t cells = wave_sum((uint64_t)slot[COUNT_CELLS]);
  const uint64_t chunks = wave_sum((uint64_t)slot[COUNT_CHUNKS]);
  if (threadIdx.x == 0) {
    out[0] = cells;
    out[1] = chunks;
  }
}

// Voxelizes runs of `per_wave` triangles, a wave each (ITEMS: the queued items
// of big triangles, one each).  A triangle's box rows go to the lanes of its
// wave, so that a wave's time follows the rows of all its triangles and not
// the largest of them, and a row costs its 15 LDS pieces and about 290
// instructions however many cells it crosses, and about 85 per four cells it
// hits.  Bound by those instructions on soups (100,000 triangles at res 1024:
// 58 us, and 24 for the queued items; a lane per triangle that tested every
// cell of its box took 216 and 75), by the atomics on small triangles
// (327,680 at res 512: 75 us, 39 without them; 110 before).
//
// Bitmap bits go through a table in LDS before they reach memory, 64 cells
// (4 x 4 x 4) an entry: an atomic on memory that all XCDs share is carried out
// beyond their L2s, about 30 G of them a second whatever their width, and
// neighboring rows and triangles set bits of the same words.  A word whose
// slot holds another goes to memory at once.  512 slots: with 1024 and 2048, or a
// second slot to try, whole builds take 0-1 % and 1-2 % longer, and the same.
constexpr uint32_t MAX_PER_WAVE = 32;
constexpr uint64_t SMALL_MAX = 1 << 20;  // cells of a triangle that shares a wave, at most
constexpr int WORD_SLOT_BITS = 9;
constexpr uint32_t WORD_SLOTS = 1u << WORD_SLOT_BITS, NO_WORD = 0xFFFFFFFFu;
struct WordTable {
  unsigned long long bits[WORD_SLOTS];
  uint32_t word[WORD_SLOTS];
};
__device__ inline void or_memory(uint32_t* bitmap, uint8_t* line_flags, uint64_t word,
                                 unsigned long long bits) {
  // (every writer of a flag stores the same value)
  if (line_flags) line_flags[word / (BITMAP_LINE_BYTES / 8)] = 1;
  __hip_atomic_fetch_or((unsigned long long*)bitmap + word, bits, __ATOMIC_RELAXED,
                        __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void set_bits(WordTable& t, uint32_t* bitmap, uint8_t* line_flags,
                                uint64_t word, unsigned long long bits) {
  if (word < NO_WORD) {
    const uint32_t slot = ((uint32_t)word * 0x9E3779B1u) >> (32 - WORD_SLOT_BITS);
    const uint32_t old = atomicCAS(&t.word[slot], NO_WORD, (uint32_t)word);
    if (old == NO_WORD || old == (uint32_t)word) {
      atomicOr(&t.bits[slot], bits);
      return;
    }
  }
  or_memory(bitmap, line_flags, word, bits);
}

template <typename K, bool BITMAP, bool ITEMS>
__global__ __launch_bounds__(BLOCK) void k_vox_rows(
    const MeshDev* meshes, const MeshParams* params, const uint64_t* tri_base, uint32_t n_meshes,
    uint64_t n_tris, int cb, uint32_t small_max, uint32_t per_wave, uint32_t scale, VoxOut<K> out,
    BigItem* big, unsigned long long* big_count, uint64_t big_cap) {
  __shared__ RowTri s_tri[WAVES][ITEMS ? 1 : MAX_PER_WAVE];
  __shared__ uint32_t s_mark[WAVES][64];
  __shared__ K s_key[BITMAP ? 1 : WAVES][BITMAP ? 1 : STAGE];
  __shared__ WordTable s_words[1];  // (bitmap path only: the key path leaves it out)
  const uint32_t w = threadIdx.x >> 6, lane = __lane_id();
  uint64_t wave = (uint64_t)blockIdx.x * WAVES + w, n_items = 0;
  if (ITEMS) {
    const uint64_t queued = *big_count;
    n_items = queued < big_cap ? queued : big_cap;
    if ((uint64_t)blockIdx.x * WAVES >= n_items) return;
  }
  if (BITMAP) {
    for (uint32_t i = threadIdx.x; i < WORD_SLOTS; i += BLOCK) {
      s_words[0].word[i] = NO_WORD;
      s_words[0].bits[i] = 0;
    }
    __syncthreads();
  }
  uint64_t n_hits = 0;      // bitmap path: this lane's
  uint32_t staged = 0;      // key path: keys in s_key (the same in every lane)
  // the code's bits of x: 0, 3, 6, ...
  constexpr K MX = (K)(sizeof(K) == 4 ? 0x09249249u : 0x1249249249249249ull);
  auto flush = [&]() {
    wave_sync();
    uint64_t base = 0;
    if (lane == 0) base = atomicAdd(out.count, (unsigned long long)staged);
    base = bcast_first(base);
    for (uint32_t i = lane; i < staged; i += 64) out.keys[base + i] = s_key[BITMAP ? 0 : w][i];
    wave_sync();
    staged = 0;
  };
  for (;;) {
    // ---- set-up: a lane per triangle
    uint64_t gid = n_tris, first = 0;
    uint32_t row0 = 0;
    bool mine;
    if (ITEMS) {
      mine = lane == 0 && wave < n_items;
      if (mine) {
        gid = big[wave].tri;
        row0 = big[wave].row0;
      }
      mine = mine && gid < n_tris;
      first = bcast_first(gid);
    } else {
      first = wave * per_wave;
      gid = first + lane;
      mine = lane < per_wave && gid < n_tris;
    }
    uint32_t rows = 0;
    const uint32_t m =
        first < n_tris ? find_mesh_wave(tri_base, n_meshes, first, mine ? gid : first) : 0u;
    {
      uint32_t chunks = 0;
      TriSetup S;
      if (mine) {
        const MeshDev& md = meshes[m];
        const MeshParams P = params[m];
        float v[3][3];
        if (P.status == 0 && load_tri(md, P, gid - md.tri_base, v)) {
          tri_setup(v, P, S);
          const uint64_t nx = S.g1[0] - S.g0[0] + 1, ny = S.g1[1] - S.g0[1] + 1,
                         nz = S.g1[2] - S.g0[2] + 1;
          if (ITEMS) {
            rows = (uint32_t)std::min<uint64_t>(BIG_ROWS, ny * nz - row0);
          } else if (nx * ny * nz <=
                     std::min<uint64_t>((uint64_t)(md.small_max ? md.small_max : small_max) * scale,
                                        SMALL_MAX)) {
            rows = (uint32_t)(ny * nz);
          } else {
            chunks = (uint32_t)((ny * nz + BIG_ROWS - 1) / BIG_ROWS);
          }
        }
      }
      if (!ITEMS && __any(chunks != 0)) {
        // one atomic per wave for its triangles' items
        const uint32_t inc = wave_incl_scan_dpp(chunks);
        uint64_t at = 0;
        if (lane == 63) at = atomicAdd(big_count, (unsigned long long)inc);
        at = (uint64_t)__shfl((uint32_t)at, 63) | ((uint64_t)__shfl((uint32_t)(at >> 32), 63) << 32);
        at += inc - chunks;
        for (uint32_t j = 0; j < chunks; ++j)
          if (at + j < big_cap) big[at + j] = BigItem{(uint32_t)gid, j * (uint32_t)BIG_ROWS};
      }
      if (rows) {
        RowTri& T = s_tri[w][ITEMS ? 0 : lane];
        row_setup(S, T);
        const uint64_t k = BITMAP ? out.bm_off[m] / 2 : (uint64_t)m << cb;  // (whole tiles)
        T.key_lo = (uint32_t)k;
        T.key_hi = (uint32_t)(k >> 32);
      }
    }
    const uint32_t inc_rows = wave_incl_scan_dpp(rows), start = inc_rows - rows;
    const uint32_t total = __builtin_amdgcn_readlane(inc_rows, 63);
    if (rows) s_tri[w][ITEMS ? 0 : lane].row0 = start - row0;
    wave_sync();
    // ---- rows: a lane each
    uint32_t owner = 0;       // 1 + the triangle of the last item taken
    for (uint32_t base = 0; base < total; base += 64) {
      const uint32_t item = base + lane;
      // the triangle of an item: triangles mark where their rows begin, and the
      // last mark at or before the item counts
      uint32_t tr = 0;
      if (!ITEMS) {
        s_mark[w][lane] = 0;
        wave_sync();
        if (rows && start >= base && start - base < 64) s_mark[w][start - base] = lane + 1;
        wave_sync();
        const uint32_t mark = s_mark[w][lane];
        owner = wave_incl_max_dpp(lane == 0 && mark == 0 ? owner : mark);
        tr = owner - 1;
        owner = __builtin_amdgcn_readlane(owner, 63);
      }
      const RowTri& T = s_tri[w][tr];
      const uint32_t r = item - T.row0;
      int y, z;
      if (ITEMS) {
        z = (int)(r / (uint32_t)T.ny);
        y = (int)(r - (uint32_t)z * (uint32_t)T.ny);
      } else {
        // r < 2^20 (SMALL_MAX), so that the quotient of
        // r + 1/2 lies at least 2^-21 of itself from a whole number: exact
        z = (int)(((float)r + 0.5f) * T.inv_ny);
        y = (int)r - z * T.ny;
      }
      y += T.y0;
      z += T.z0;
      int xa = 0, xb = -1, ia = 0, ib = -1;
      RowTerms R;
      if (item < total && row_terms(T, y, z, R)) row_range(T, R, xa, xb, ia, ib);
      // four cells at a time: they share a bitmap word
      const uint64_t kbase = (uint64_t)T.key_lo | ((uint64_t)T.key_hi << 32);
      int x = xa & ~3;
      K code = morton3<K>((uint32_t)x, (uint32_t)y, (uint32_t)z);
      while (__any(x <= xb)) {
        uint32_t hit = 0, test = 0;
        if (x <= xb) {
          // bits [a, b] of four
          auto span = [&](int a, int b) -> uint32_t {
            a = a > x ? a - x : 0;
            b = b < x + 3 ? b - x : 3;
            return a <= b ? (2u << b) - (1u << a) : 0u;
          };
          test = span(xa, xb);
          hit = span(ia, ib) & test;
          test &= ~hit;
        }
        while (__any(test != 0)) {  // cells that rounding could decide either way
          if (test) {
            const uint32_t j = __builtin_ctz(test);
            if (cell_hit(T, R, x + (int)j)) hit |= 1u << j;
            test &= test - 1u;
          }
        }
        if (BITMAP) {
          if (hit) {
            n_hits += __popc(hit);
            // cells 0-3 of the group are bits 0, 1, 8, 9 from its place
            set_bits(s_words[0], out.bits, out.line_flags, kbase + (uint64_t)(code >> 6),
                     (unsigned long long)((hit & 3u) | ((hit & 12u) << 6)) << (code & 63));
          }
        } else {
          const uint32_t cnt = __popc(hit), inc = wave_incl_scan_dpp(cnt);
          uint32_t at = staged + inc - cnt;
          for (uint32_t h = hit; h; h &= h - 1u) {
            const uint32_t j = __builtin_ctz(h);
            s_key[BITMAP ? 0 : w][at++] = (K)kbase | code | (K)((j & 1u) | ((j & 2u) << 2));
          }
          staged += __builtin_amdgcn_readlane(inc, 63);
          if (staged > STAGE - 256) flush();
        }
        x += 4;
        // x + 4 in the code: one added to the bits of x from bit 2 on (bits 0 and
        // 1 are zero), the others set so that the carry passes them
        constexpr K M4 = MX & ~(K)9;
        code = (((code | ~M4) + 1) & M4) | (code & ~M4);
      }
    }
    wave += (uint64_t)gridDim.x * WAVES;
    if (!ITEMS || wave >= n_items) break;
    wave_sync();  // s_tri is written again
  }
  if (BITMAP) {
    uint32_t h = (uint32_t)n_hits;  // a lane's rows hold fewer than 2^32 cells
    h = wave_sum_u32(h);
    if (h && lane == 0)
      atomicAdd(out.slots + (wave % COUNT_SLOTS) * COUNT_STRIDE + COUNT_HITS, (unsigned long long)h);
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < WORD_SLOTS; i += BLOCK)
      if (s_words[0].word[i] != NO_WORD)
        or_memory(out.bits, out.line_flags, s_words[0].word[i], s_words[0].bits[i]);
  } else if (staged) {
    flush();
  }
}

}  // namespace

void launch_begin(const PassBegin& B, hipStream_t s) {
  const uint64_t n = std::max({B.n_table, B.n_zero, (uint64_t)B.n_meshes * 8});
  const uint64_t blocks = std::min<uint64_t>((n + BLOCK - 1) / BLOCK, 1024);
  hipLaunchKernelGGL(k_begin, dim3((uint32_t)std::max<uint64_t>(blocks, 1)), dim3(BLOCK), 0, s, B);
}

void launch_bbox(const MeshDev* meshes, uint32_t n_meshes, uint64_t max_points, uint64_t max_tris,
                 uint32_t* acc, hipStream_t s) {
  const auto blocks = [](uint64_t n) {
    return (uint32_t)std::min<uint64_t>((3 * n + FLAT_CHUNK - 1) / FLAT_CHUNK, BBOX_BLOCKS);
  };
  const uint32_t pb = blocks(max_points), tb = blocks(max_tris);
  if (pb + tb == 0) return;
  hipLaunchKernelGGL(k_bbox, dim3(pb + tb, n_meshes), dim3(BLOCK), 0, s, meshes, pb, acc);
}

void launch_classify(const MeshDev* meshes, const uint32_t* acc, MeshParams* params,
                     const uint64_t* tri_base, uint32_t n_meshes, uint64_t n_tris,
                     const Tuning& tn, unsigned long long* slots, hipStream_t s) {
  const uint64_t blocks = (std::max<uint64_t>(n_tris, n_meshes) + BLOCK - 1) / BLOCK;
  hipLaunchKernelGGL(k_classify, dim3((uint32_t)std::min<uint64_t>(blocks, CLASSIFY_BLOCKS)),
                     dim3(BLOCK), 0, s, meshes, acc, params, tri_base, n_meshes, n_tris,
                     tn.small_max_cells, slots);
}

void launch_read_totals(const unsigned long long* slots, unsigned long long* out, hipStream_t s) {
  hipLaunchKernelGGL(k_read_totals, dim3(1), dim3(COUNT_SLOTS), 0, s, slots, out);
}

template <typename K, bool BITMAP>
static void launch_rows(const MeshDev* meshes, const MeshParams* params, const uint64_t* tri_base,
                        uint32_t n_meshes, uint64_t n_tris, int cb, const Tuning& tn,
                        const VoxOut<K>& out, BigItem* big, unsigned long long* big_count,
                        uint64_t big_cap, hipStream_t s) {
  // triangles per wave: 32 while that leaves 8 waves to each of the 1024
  // SIMDs, fewer in smaller passes (at least 4: a wave sets up as many
  // triangles at a time as it has).  Waves that stage keys take as many as
  // leaves 2 to a SIMD: each reserves its keys' places at least once, and
  // atomics on the one key count follow each other at about 6 ns.
  uint32_t per = MAX_PER_WAVE;
  while (per > 4 && n_tris / per < (BITMAP ? 8192 : 2048)) per /= 2;
  // The size limit is that of triangles that share a wave by 16 or 32; where
  // fewer do, as many times larger ones may (100,000 triangles, 8 to a wave,
  // limits of 1024 / 2048 / 4096 cells: 269 / 214 / 189 us at 2048^3, 83 / 85 /
  // 94 at 1024^3; the batch's coarse meshes, 32 to a wave: 306 / 354 / 528).  A
  // queued item costs a wave that stages keys its own place in the output, so
  // that these take twice the limit (sparse hits at 4096^3: 255 / 199 / 203).
  // The classification counts the items with the limit itself: a bound.
  const uint32_t scale = std::max(1u, MAX_PER_WAVE / 2 / per) * (BITMAP ? 1 : 2);
  const uint64_t waves = (n_tris + per - 1) / per;
  hipLaunchKernelGGL((k_vox_rows<K, BITMAP, false>), dim3((uint32_t)((waves + WAVES - 1) / WAVES)),
                     dim3(BLOCK), 0, s, meshes, params, tri_base, n_meshes, n_tris, cb,
                     tn.small_max_cells, per, scale, out, big, big_count, big_cap);
  if (big_cap)
    hipLaunchKernelGGL((k_vox_rows<K, BITMAP, true>),
                       dim3((uint32_t)std::min<uint64_t>((big_cap + WAVES - 1) / WAVES, BIG_BLOCKS)),
                       dim3(BLOCK), 0, s, meshes,
                       params, tri_base, n_meshes, n_tris, cb, tn.small_max_cells, 1u, 1u, out, big,
                       big_count, big_cap);
}

template <typename K>
void launch_voxelize(const MeshDev* meshes, const MeshParams* params, const uint64_t* tri_base,
                     uint32_t n_meshes, uint64_t n_tris, int cb, const Tuning& tn, K* keys,
                     uint32_t* bitmap, const uint64_t* bm_off, uint8_t* line_flags,
                     unsigned long long* key_count, unsigned long long* slots, BigItem* big,
                     unsigned long long* big_count, uint64_t big_cap, hipStream_t s) {
  if (n_tris == 0) return;
  const VoxOut<K> out{keys, bitmap, bm_off, line_flags, key_count, slots};
  if (bitmap)
    launch_rows<K, true>(meshes, params, tri_base, n_meshes, n_tris, cb, tn, out, big, big_count,
                         big_cap, s);
  else
    launch_rows<K, false>(meshes, params, tri_base, n_meshes, n_tris, cb, tn, out, big, big_count,
                          big_cap, s);
}

template void launch_voxelize<uint32_t>(const MeshDev*, const MeshParams*, const uint64_t*,
                                        uint32_t, uint64_t, int, const Tuning&, uint32_t*,
                                        uint32_t*, const uint64_t*, uint8_t*,
                                        unsigned long long*,
                                        unsigned long long*, BigItem*, unsigned long long*,
                                        uint64_t, hipStream_t);
template void launch_voxelize<uint64_t>(const MeshDev*, const MeshParams*, const uint64_t*,
                                        uint32_t, uint64_t, int, const Tuning&, uint64_t*,
                                        uint32_t*, const uint64_t*, uint8_t*,
                                        unsigned long long*,
                                        unsigned long long*, BigItem*, unsigned long long*,
                                        uint64_t, hipStream_t);

}  // namespace svo
