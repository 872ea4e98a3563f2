// Exact k-nearest-neighbour search on gfx950.
//
// Replaces the reference's grid kNN (knearests.cu:19-145, 230-386) and its
// brute-force kNN (extern/kNN-CUDA/knncuda.cu:20-91, 143-189, 271-349).
//
// Result contract: for every query, the k reference points with the smallest
// (d2, index) keys, nearest first, where d2 = fma(dz,dz, fma(dy,dy, dx*dx)) in
// FP32 with d = ref - query.  The output does not depend on the grid, the
// launch shape or the order of work, so it is bit-exact against any exact
// implementation that uses the same key.
//
// Grid: a uniform grid over the bounding box of the reference points (and an
// optional extra box), sized on the device so that a whole Lloyd iteration can
// be captured in a graph.  Binning is a counting sort (count, scan, scatter)
// followed by an in-cell sort by index, so the sorted order is deterministic.
//
// Query: one wavefront per query.  The wave walks a table of cell offsets
// ordered by a query-independent lower bound of their distance, loads the
// points of 64 cells at a time into its 64 lanes, filters them against the
// current k-th key, stages survivors in LDS and merges every 64 of them into a
// sorted top-k held in registers (64*M slots, bitonic sort + bitonic merge
// across lanes).  It stops when the lower bound of the next offsets exceeds
// the k-th distance; offsets beyond the table fall back to a full scan.
#include "vd_knn.hpp"

#include <algorithm>
#include <climits>
#include <cmath>
#include <vector>

namespace vd {

namespace {

constexpr int kScanThreads = 1024;

__device__ __forceinline__ int cell_coord(float x, float lo, float inv_h, int dim) {
  int c = (int)floorf((x - lo) * inv_h);
  return min(max(c, 0), dim - 1);
}

__device__ __forceinline__ uint32_t bperm32(uint32_t v, int src_lane) {
  return (uint32_t)__builtin_amdgcn_ds_bpermute(src_lane << 2, (int)v);
}
__device__ __forceinline__ uint64_t bperm64(uint64_t v, int src_lane) {
  const uint32_t lo = bperm32((uint32_t)v, src_lane);
  const uint32_t hi = bperm32((uint32_t)(v >> 32), src_lane);
  return ((uint64_t)hi << 32) | lo;
}

// Value of lane (lane ^ j) for a compile-time j: within a row of 16 lanes
// through DPP moves (quad permutes for 1 and 2; row rotations, where lane i
// reads lane i - n of its row, for 4 and 8), which stay in the VALU, and
// through the LDS crossbar (ds_bpermute) for 16 and 32.
__device__ __forceinline__ uint32_t xor_lane32(uint32_t v, int j, int lane) {
  const int x = (int)v;
  switch (j) {
    case 1: return (uint32_t)__builtin_amdgcn_mov_dpp(x, 0xB1, 0xF, 0xF, false);   // quad_perm [1,0,3,2]
    case 2: return (uint32_t)__builtin_amdgcn_mov_dpp(x, 0x4E, 0xF, 0xF, false);   // quad_perm [2,3,0,1]
    case 4: {
      // lanes without bit 2 (banks 0 and 2 of a row): row_ror:12, lane i + 4;
      // then the others (banks 1 and 3): row_ror:4, lane i - 4
      const int from_above = __builtin_amdgcn_mov_dpp(x, 0x12C, 0xF, 0x5, false);
      return (uint32_t)__builtin_amdgcn_update_dpp(from_above, x, 0x124, 0xF, 0xA, false);
    }
    case 8: return (uint32_t)__builtin_amdgcn_mov_dpp(x, 0x128, 0xF, 0xF, false);  // row_ror:8
    default: return bperm32(v, lane ^ j);
  }
}
__device__ __forceinline__ uint64_t xor_lane64(uint64_t v, int j, int lane) {
  const uint32_t lo = xor_lane32((uint32_t)v, j, lane);
  const uint32_t hi = xor_lane32((uint32_t)(v >> 32), j, lane);
  return ((uint64_t)hi << 32) | lo;
}

// Inclusive prefix sum across the wave through DPP moves: row shifts by 1, 2,
// 4 and 8 within each row of 16 lanes (lanes without a source add 0), then
// the last lane of row 0 into row 1 and of row 2 into row 3 (row_bcast:15),
// then the last lane of row 1 into rows 2 and 3 (row_bcast:31).
__device__ __forceinline__ int wave_incl_sum(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, false);  // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, false);  // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, false);  // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, false);  // row_shr:8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xA, 0xF, false);  // row_bcast:15, rows 1 and 3
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xC, 0xF, false);  // row_bcast:31, rows 2 and 3
  return x;
}
// Inclusive prefix maximum across the wave, the same DPP steps (lanes
// without a source contribute -1).
__device__ __forceinline__ int wave_incl_max(int x) {
  x = max(x, __builtin_amdgcn_update_dpp(-1, x, 0x111, 0xF, 0xF, false));
  x = max(x, __builtin_amdgcn_update_dpp(-1, x, 0x112, 0xF, 0xF, false));
  x = max(x, __builtin_amdgcn_update_dpp(-1, x, 0x114, 0xF, 0xF, false));
  x = max(x, __builtin_amdgcn_update_dpp(-1, x, 0x118, 0xF, 0xF, false));
  x = max(x, __builtin_amdgcn_update_dpp(-1, x, 0x142, 0xA, 0xF, false));
  x = max(x, __builtin_amdgcn_update_dpp(-1, x, 0x143, 0xC, 0xF, false));
  return x;
}

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Owner lane of flat index f0 + lane of the cells' concatenated point ranges
// (the largest lane whose range starts at or before it): every lane with
// points whose range starts in [f0, f0 + 64) marks its start in `mark`, a
// prefix maximum over the marks finds the latest start, and `carry` (the
// owner of f0 - 1, 0 at first) covers ranges begun in earlier batches.
__device__ __forceinline__ int batch_owner(int* mark, int lane, int cnt, int excl, int f0, int& carry) {
  mark[lane] = -1;
  wave_sync();
  if (cnt > 0 && excl >= f0 && excl < f0 + 64) mark[excl - f0] = lane;
  wave_sync();
  const int own = max(wave_incl_max(mark[lane]), carry);
  carry = __builtin_amdgcn_readlane(own, 63);
  wave_sync();
  return own;
}
__device__ __forceinline__ uint64_t umin64(uint64_t a, uint64_t b) { return a < b ? a : b; }

// A key orders by (d2, id): the bits of d2 >= 0 (every NaN taken as the same
// one, after infinity) plus kKeyShift in the high word, the id in the low one.
// As a double it is positive, finite and normal (the shift lifts it out of the
// subnormals, and the largest high word, of a NaN, is below the exponent of
// infinity), so the order of the keys is the order of the doubles, and one
// v_min_f64 takes the smaller of two keys unchanged where a 64-bit integer
// compare needs two selects after it.  kNoKey, larger than every key, is an
// empty place.
constexpr uint32_t kKeyShift = 0x00100000u;
constexpr uint64_t kNoKey = 0x7FEFFFFFFFFFFFFFull;
__device__ __forceinline__ uint32_t key_word(float d2) { return min(__float_as_uint(d2), 0x7FC00000u) + kKeyShift; }
__device__ __forceinline__ uint64_t knn_key(float d2, uint32_t id) { return ((uint64_t)key_word(d2) << 32) | id; }
// The largest key at distance d2.
__device__ __forceinline__ uint64_t key_bound(float d2) { return ((uint64_t)key_word(d2) << 32) | 0xffffffffull; }
__device__ __forceinline__ float key_d2(uint64_t k) { return __uint_as_float((uint32_t)(k >> 32) - kKeyShift); }

// min(a, b), max(a, b) and min(a, -b) of keys and negated keys (sign bit set).
// The s_nop is the distance that a VALU result needs before a DPP move reads
// it, which the compiler does not add behind inline assembly.
__device__ __forceinline__ uint64_t key_min(uint64_t a, uint64_t b) {
  uint64_t r;
  asm("v_min_f64 %0, %1, %2\n\ts_nop 1" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ uint64_t key_max(uint64_t a, uint64_t b) {
  uint64_t r;
  asm("v_max_f64 %0, %1, %2\n\ts_nop 1" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ uint64_t key_min_neg(uint64_t a, uint64_t b) {
  uint64_t r;
  asm("v_min_f64 %0, %1, -%2\n\ts_nop 1" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
// x with its sign bit flipped where `sign` (0 or 0x80000000) says so.
__device__ __forceinline__ uint64_t flip(uint64_t x, uint32_t sign) { return x ^ ((uint64_t)sign << 32); }

__device__ __forceinline__ float dist2(const float4& r, const float4& q) {
  const float dx = r.x - q.x, dy = r.y - q.y, dz = r.z - q.z;
  return fmaf(dz, dz, fmaf(dy, dy, dx * dx));
}

// ---------------------------------------------------------------- grid ----

// Bounding box of points p0..p1 over the workgroup, a part per wave in red.
__device__ __forceinline__ void points_box(const float4* pts, int p0, int p1, float (*red)[kScanThreads / 64]) {
  float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
  for (int i = p0 + threadIdx.x; i < p1; i += blockDim.x) {
    const float4 p = pts[i];
    lo[0] = fminf(lo[0], p.x); lo[1] = fminf(lo[1], p.y); lo[2] = fminf(lo[2], p.z);
    hi[0] = fmaxf(hi[0], p.x); hi[1] = fmaxf(hi[1], p.y); hi[2] = fmaxf(hi[2], p.z);
  }
  for (int off = 32; off > 0; off >>= 1)
    for (int a = 0; a < 3; ++a) {
      lo[a] = fminf(lo[a], __shfl_xor(lo[a], off));
      hi[a] = fmaxf(hi[a], __shfl_xor(hi[a], off));
    }
  if ((threadIdx.x & 63) == 0)
    for (int a = 0; a < 3; ++a) {
      red[a][threadIdx.x >> 6] = lo[a];
      red[3 + a][threadIdx.x >> 6] = hi[a];
    }
  __syncthreads();
}
__device__ __forceinline__ void join_boxes(float (*red)[kScanThreads / 64], float lo[3], float hi[3]) {
  for (int a = 0; a < 3; ++a) {
    lo[a] = red[a][0];
    hi[a] = red[3 + a][0];
    for (int j = 1; j < (int)(blockDim.x >> 6); ++j) {
      lo[a] = fminf(lo[a], red[a][j]);
      hi[a] = fmaxf(hi[a], red[3 + a][j]);
    }
  }
}

// Grid shape of n points with bounding box lo..hi, which it extends by the box
// extra_lo..extra_hi (use_extra): about n/density cells of equal size, at most
// max_cells.
__device__ GridShape make_shape(const float lo[3], const float hi[3], const float3& extra_lo, const float3& extra_hi,
                                int use_extra, int n, float density, int max_cells) {
  double l[3], h[3];
  const float elo[3] = {extra_lo.x, extra_lo.y, extra_lo.z}, ehi[3] = {extra_hi.x, extra_hi.y, extra_hi.z};
  for (int a = 0; a < 3; ++a) {
    l[a] = lo[a];
    h[a] = hi[a];
    if (use_extra) {
      l[a] = fmin(l[a], (double)elo[a]);
      h[a] = fmax(h[a], (double)ehi[a]);
    }
    if (!(l[a] <= h[a])) { l[a] = 0.0; h[a] = 0.0; }
  }
  double ext = fmax(fmax(h[0] - l[0], h[1] - l[1]), fmax(h[2] - l[2], 1e-20));
  // pad the box so that no point sits on the upper face
  for (int a = 0; a < 3; ++a) {
    l[a] -= 1e-4 * ext;
    h[a] += 1e-4 * ext;
  }
  ext *= 1.0002;
  double vol = 1.0;
  for (int a = 0; a < 3; ++a) vol *= fmax(h[a] - l[a], ext * 1e-3);
  const double cells = fmax(1.0, (double)n / (double)density);
  double cs = cbrt(vol / cells);
  int dim[3];
  for (;;) {
    long long tot = 1;
    for (int a = 0; a < 3; ++a) {
      dim[a] = (int)fmin(1024.0, fmax(1.0, ceil((h[a] - l[a]) / cs)));
      tot *= dim[a];
    }
    if (tot <= max_cells) break;
    cs *= 1.05;
  }
  GridShape g;
  for (int a = 0; a < 3; ++a) {
    g.lo[a] = (float)l[a];
    g.dim[a] = dim[a];
  }
  g.h = (float)cs;
  g.inv_h = (float)(1.0 / cs);
  g.ncell = dim[0] * dim[1] * dim[2];
  // absolute slack for the cell-box distance bounds (rounding of the cell
  // assignment and of lo + c*h)
  g.slack = (float)(1e-3 * cs + 1e-6 * (fabs(l[0]) + fabs(l[1]) + fabs(l[2]) + 1024.0 * cs));
  return g;
}

// Bounding boxes of the n points' parts, one workgroup each, for
// k_grid_shape's `parts` (6 floats per workgroup).
constexpr int kBoxParts = 64;
__global__ __launch_bounds__(kScanThreads) void k_grid_box(const float4* pts, int n, float* parts) {
  __shared__ float red[6][kScanThreads / 64];
  const int per = (n + (int)gridDim.x - 1) / (int)gridDim.x;
  const int p0 = min(n, (int)blockIdx.x * per);
  points_box(pts, p0, min(n, p0 + per), red);
  if (threadIdx.x == 0) {
    float lo[3], hi[3];
    join_boxes(red, lo, hi);
    for (int a = 0; a < 3; ++a) {
      parts[6 * blockIdx.x + a] = lo[a];
      parts[6 * blockIdx.x + 3 + a] = hi[a];
    }
  }
}

// The grid shape over the points' bounding box (and `extra`, a box given by
// the host); one block per instance.  The single instance may give the boxes
// of its points' parts (k_grid_box) instead of having one workgroup read all
// points (100,000: 41 us -> 11 for both kernels; 200,000: 90 -> 11).
__global__ __launch_bounds__(kScanThreads) void k_grid_shape(const float4* pts, int n, const int* pt_begin,
                                                              const int* cell_base, const float* box, float3 extra_lo,
                                                              float3 extra_hi, int use_extra, float density,
                                                              int max_cells, const float* parts, int n_parts,
                                                              GridShape* shapes) {
  __shared__ float red[6][kScanThreads / 64];
  const int inst = blockIdx.x;
  const int p0 = pt_begin ? pt_begin[inst] : 0, p1 = pt_begin ? pt_begin[inst + 1] : n;
  if (cell_base) max_cells = cell_base[inst + 1] - cell_base[inst];
  if (box) {
    extra_lo = make_float3(box[6 * inst], box[6 * inst + 1], box[6 * inst + 2]);
    extra_hi = make_float3(box[6 * inst + 3], box[6 * inst + 4], box[6 * inst + 5]);
    use_extra = 1;
  }
  float lo[3], hi[3];
  if (parts) {  // one wave
    const int lane = threadIdx.x;
    for (int a = 0; a < 3; ++a) {
      lo[a] = lane < n_parts ? parts[6 * lane + a] : INFINITY;
      hi[a] = lane < n_parts ? parts[6 * lane + 3 + a] : -INFINITY;
      for (int off = 32; off > 0; off >>= 1) {
        lo[a] = fminf(lo[a], __shfl_xor(lo[a], off));
        hi[a] = fmaxf(hi[a], __shfl_xor(hi[a], off));
      }
    }
  } else {
    points_box(pts, p0, p1, red);
  }
  if (threadIdx.x == 0) {
    if (!parts) join_boxes(red, lo, hi);
    shapes[inst] = make_shape(lo, hi, extra_lo, extra_hi, use_extra, p1 - p0, density, max_cells);
  }
}

__global__ void k_grid_count(const float4* pts, int n, const GridShape* gs, const int* pt_inst, const int* cell_base,
                             int* cell_of, int* count) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int inst = pt_inst ? pt_inst[i] : 0;
  const GridShape g = gs[inst];
  const float4 p = pts[i];
  const int cx = cell_coord(p.x, g.lo[0], g.inv_h, g.dim[0]);
  const int cy = cell_coord(p.y, g.lo[1], g.inv_h, g.dim[1]);
  const int cz = cell_coord(p.z, g.lo[2], g.inv_h, g.dim[2]);
  const int c = (cell_base ? cell_base[inst] : 0) + cx + g.dim[0] * (cy + g.dim[1] * cz);
  cell_of[i] = c;
  atomicAdd(count + c, 1);
}

__global__ void k_grid_scatter(int n, const int* cell_of, const int* start, int* cursor, int* sorted_ids) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int c = cell_of[i];
  sorted_ids[start[c] + atomicAdd(cursor + c, 1)] = i;
}

// Orders every cell's points by index: each point's place is the number of
// smaller ids in its cell, so the loads of a cell do not depend on each other.
// sorted_pts gets the points (their ids in w) and then sorted_ids the ids.  A
// workgroup takes kSortCells cells: a lane of its first wave a cell of at most
// kLightCell points, and the workgroup together each fuller one.  (One lane
// inserting a cell's ids one by one took 4.3 ms at 200,000 clustered sites,
// where a cell holds up to a few thousand; one wave per heavy cell 0.45 ms;
// this 0.11 ms.)
// n_cells < 0: the cells of the single instance gs[0].
constexpr int kLightCell = 16, kSortCells = 64, kSortThreads = 256, kSortTile = 1024;
__device__ __forceinline__ float4 with_id(float4 p, int id) {
  p.w = __int_as_float(id);
  return p;
}
__global__ __launch_bounds__(kSortThreads) void k_grid_sort(const GridShape* gs, int n_cells, const float4* pts,
                                                            const int* start, int* sorted_ids, float4* sorted_pts) {
  __shared__ int4 tile[kSortTile / 4];
  __shared__ int heavy_b[kSortCells], heavy_e[kSortCells];
  __shared__ int n_heavy;
  const int tid = threadIdx.x;
  int b = 0, e = 0;
  if (tid < kSortCells) {
    const int c = blockIdx.x * kSortCells + tid;
    if (c < (n_cells >= 0 ? n_cells : gs->ncell)) {
      b = start[c];
      e = start[c + 1];
    }
    const bool heavy = e - b > kLightCell;
    const uint64_t m = __ballot(heavy);
    if (heavy) {
      const int k = __popcll(m & ((1ull << tid) - 1ull));
      heavy_b[k] = b;
      heavy_e[k] = e;
      b = e;
    }
    if (tid == 0) n_heavy = __popcll(m);
    for (int i = b; i < e; ++i) {
      const int v = sorted_ids[i];
      int rank = 0;
      for (int j = b; j < e; ++j) rank += sorted_ids[j] < v;
      sorted_pts[b + rank] = with_id(pts[v], v);
    }
  }
  __syncthreads();
  for (int h = 0; h < n_heavy; ++h) {
    const int hb = heavy_b[h], he = heavy_e[h];
    for (int i0 = hb; i0 < he; i0 += kSortThreads) {
      const int i = i0 + tid;
      const int v = i < he ? sorted_ids[i] : INT_MAX;
      int rank = 0;
      for (int t0 = hb; t0 < he; t0 += kSortTile) {
        __syncthreads();
        for (int j = tid; j < kSortTile; j += kSortThreads)
          ((int*)tile)[j] = t0 + j < he ? sorted_ids[t0 + j] : INT_MAX;
        __syncthreads();
        const int n4 = (min(kSortTile, he - t0) + 3) / 4;
        for (int j = 0; j < n4; ++j) {
          const int4 q = tile[j];
          rank += (q.x < v) + (q.y < v) + (q.z < v) + (q.w < v);
        }
      }
      if (i < he) sorted_pts[hb + rank] = with_id(pts[v], v);
    }
  }
  __threadfence_block();
  __syncthreads();
  if (tid < kSortCells)
    for (int i = b; i < e; ++i) sorted_ids[i] = __float_as_int(sorted_pts[i].w);
  for (int h = 0; h < n_heavy; ++h)
    for (int i = heavy_b[h] + tid; i < heavy_e[h]; i += kSortThreads) sorted_ids[i] = __float_as_int(sorted_pts[i].w);
}

// The whole grid build of an instance of at most kSmallPoints points and
// kSmallCells cells in one workgroup, with the cell counts and the ids in LDS:
// box and shape, counts, scan, scatter, order in the cells.  One launch
// instead of eight, whose latencies are all that small problems pay (1,037
// points: 43 us -> 9.3; 131: 42 -> 7.6).  The limit is what the LDS holds with
// room to spare; at 3,001 points the one workgroup takes 17 us (the eight
// launches 43).  The tables are those of the other path.
constexpr int kSmallPoints = 8192, kSmallCells = 8192;
__global__ __launch_bounds__(kScanThreads) void k_grid_small(const float4* pts, int n, const int* pt_begin,
                                                              const int* cell_base, const float* box, float3 extra_lo,
                                                              float3 extra_hi, int use_extra, float density,
                                                              int max_cells, int n_inst, GridShape* shapes, int* count,
                                                              int* start, int* sorted_ids, float4* sorted_pts) {
  __shared__ float red[6][kScanThreads / 64];
  __shared__ int wsum[kScanThreads / 64];
  __shared__ GridShape g;
  __shared__ int cnt[kSmallCells];
  __shared__ int ids[kSmallPoints];
  const int inst = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int p0 = pt_begin ? pt_begin[inst] : 0, p1 = pt_begin ? pt_begin[inst + 1] : n;
  const int c0 = cell_base ? cell_base[inst] : 0;
  const int cells = (cell_base ? cell_base[inst + 1] : max_cells) - c0;
  const int np = p1 - p0;
  if (box) {
    extra_lo = make_float3(box[6 * inst], box[6 * inst + 1], box[6 * inst + 2]);
    extra_hi = make_float3(box[6 * inst + 3], box[6 * inst + 4], box[6 * inst + 5]);
    use_extra = 1;
  }
  points_box(pts, p0, p1, red);
  if (tid == 0) {
    float lo[3], hi[3];
    join_boxes(red, lo, hi);
    g = make_shape(lo, hi, extra_lo, extra_hi, use_extra, np, density, cells);
    shapes[inst] = g;
  }
  for (int i = tid; i < cells; i += kScanThreads) cnt[i] = 0;
  __syncthreads();
  auto cell_at = [&](const float4& p) {
    const int cx = cell_coord(p.x, g.lo[0], g.inv_h, g.dim[0]);
    const int cy = cell_coord(p.y, g.lo[1], g.inv_h, g.dim[1]);
    const int cz = cell_coord(p.z, g.lo[2], g.inv_h, g.dim[2]);
    return cx + g.dim[0] * (cy + g.dim[1] * cz);
  };
  for (int i = tid; i < np; i += kScanThreads) atomicAdd(&cnt[cell_at(pts[p0 + i])], 1);
  __syncthreads();
  // exclusive scan of the counts, kPer consecutive cells per thread
  constexpr int kPer = kSmallCells / kScanThreads;
  int v[kPer], sum = 0;
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int c = tid * kPer + k;
    v[k] = c < cells ? cnt[c] : 0;
    sum += v[k];
  }
  const int incl = wave_incl_sum(sum);
  if (lane == 63) wsum[wv] = incl;
  __syncthreads();
  int run = incl - sum;
  for (int w = 0; w < wv; ++w) run += wsum[w];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int c = tid * kPer + k;
    if (c < cells) {
      count[c0 + c] = v[k];
      start[c0 + c] = p0 + run;
      cnt[c] = run;
    }
    run += v[k];
  }
  if (inst == n_inst - 1 && tid == 0) start[c0 + cells] = p1;
  __syncthreads();
  for (int i = tid; i < np; i += kScanThreads) ids[atomicAdd(&cnt[cell_at(pts[p0 + i])], 1)] = p0 + i;
  __syncthreads();
  // cnt[c] is now the end of cell c, so its start is the end of cell c - 1
  for (int i = tid; i < np; i += kScanThreads) {
    const int id = ids[i];
    const float4 p = pts[id];
    const int c = cell_at(p);
    const int b = c > 0 ? cnt[c - 1] : 0, e = cnt[c];
    int rank = 0;
    for (int j = b; j < e; ++j) rank += ids[j] < id;
    sorted_ids[p0 + b + rank] = id;
    sorted_pts[p0 + b + rank] = with_id(p, id);
  }
}

// ---------------------------------------------------------------- query ---

struct QueryArgs {
  const GridShape* grid;  // per instance
  const int* cell_base;   // per instance, or null (one instance)
  const int* pt_inst;     // instance of every point, or null
  const int* q_inst;      // modes 1 and 2: instance of every query, or null
  const float4* sorted_pts;
  const int* sorted_ids;
  const int* start;
  int n_ref;
  const int4* offsets;  // (dx, dy, dz, lb) sorted by lb = sum max(|d|-1,0)^2
  int n_offsets;
  int k;
  int n_query;
  int mode;  // 0: queries are the reference points themselves (self excluded)
             // 1: queries are tet centroids
             // 2: queries are given points (self not excluded)
             // 3: queries are the points qpts[q_ids[q]] with ids q_ids[q] (self excluded)
  const int* q_ids;
  const unsigned* n_query_dev;  // optional device count, capping n_query
  const float4* verts;
  const int4* tets;
  const float4* qpts;
  int32_t* out;        // row-major n_query x k, or pitched rows when pitch > 0
  long long out_pitch; // > 0: out[j * pitch + q] (column per query)
  // modes 0 and 1 with row-major output: when hint_pts is given, every row of
  // `out` holds a previous result of this problem (k distinct reference ids of
  // the query's instance, the query itself excluded) and hint_pts holds the
  // reference points by original id
  const float4* hint_pts;
  const int* pt_begin;  // first point of every instance (n_inst + 1), or null
  int run;              // consecutive queries per wave (launch_query)
};

template <int M>
struct TopK {
  uint64_t s[M];
};

// The sorting networks keep a lane's key negated where the lane takes the
// larger key of its pair: with partner's value o, which has the other sign,
// min(x, -o) is then the step for both lanes of a pair, one instruction after
// the move, and the sign flips between two steps by a mask that the lane
// number gives (two compares and six selects per step without it; kNN phase
// at 1M tets / 100,000 sites 1.84 -> 1.56 ms).
//
// Sign bit of bit i of the lane number.
__device__ __forceinline__ uint32_t lane_sign(int lane, int i) { return ((uint32_t)lane << (31 - i)) & 0x80000000u; }

// Bitonic sort of one key per lane across the wave, ascending, or descending
// with desc = 0x80000000 (wave-uniform).  In the step (k, j) the lanes whose
// bits j and k differ take the larger key.
__device__ __forceinline__ uint64_t wave_sort64(uint64_t x, int lane, uint32_t desc) {
  x = flip(x, lane_sign(lane, 0) ^ lane_sign(lane, 1) ^ desc);
#pragma unroll
  for (int k = 1; k <= 6; ++k) {
#pragma unroll
    for (int j = k - 1; j >= 0; --j) {
      x = key_min_neg(x, xor_lane64(x, 1 << j, lane));
      if (j > 0)
        x = flip(x, lane_sign(lane, j) ^ lane_sign(lane, j - 1));
      else if (k < 5)
        x = flip(x, lane_sign(lane, 0) ^ lane_sign(lane, k + 1));
      else if (k == 5)
        x = flip(x, lane_sign(lane, 0));
    }
  }
  return flip(x, lane_sign(lane, 0) ^ desc);
}

// Sorted merge of 64 new keys (one per lane) into the top list; into an
// empty list (first) the sorted keys are the list.
template <int M>
__device__ __forceinline__ void topk_merge(TopK<M>& L, uint64_t x, int lane, bool first = false) {
  x = wave_sort64(x, lane, first ? 0u : 0x80000000u);
  if (first) {
    L.s[0] = x;
    return;
  }
  // min against the descending batch gives the 64*M smallest as a bitonic sequence
  L.s[M - 1] = key_min(L.s[M - 1], x);
#pragma unroll
  for (int js = M / 2; js >= 1; js >>= 1) {
#pragma unroll
    for (int s = 0; s < M; ++s) {
      if ((s & js) == 0) {
        const uint64_t a = L.s[s], b = L.s[s + js];
        L.s[s] = key_min(a, b);
        L.s[s + js] = key_max(a, b);
      }
    }
  }
#pragma unroll
  for (int s = 0; s < M; ++s) L.s[s] = flip(L.s[s], lane_sign(lane, 5));
#pragma unroll
  for (int j = 5; j >= 0; --j) {
#pragma unroll
    for (int s = 0; s < M; ++s) {
      const uint64_t m = key_min_neg(L.s[s], xor_lane64(L.s[s], 1 << j, lane));
      L.s[s] = flip(m, j > 0 ? lane_sign(lane, j) ^ lane_sign(lane, j - 1) : lane_sign(lane, 0));
    }
  }
}

template <int M>
__device__ __forceinline__ uint64_t topk_kth(const TopK<M>& L, int k) {
  const int slot = (k - 1) >> 6, ln = (k - 1) & 63;
  uint64_t v = 0;
#pragma unroll
  for (int s = 0; s < M; ++s)
    if (s == slot) v = L.s[s];
  const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)v, ln);
  const uint32_t hi = __builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), ln);
  return ((uint64_t)hi << 32) | lo;
}

// Inserts one key (wave-uniform) into the sorted list: the keys after its
// place move up one slot and the largest drops out.
template <int M>
__device__ __forceinline__ void topk_insert(TopK<M>& L, uint64_t x, int lane) {
  int pos = 0;
#pragma unroll
  for (int s = 0; s < M; ++s) pos += __popcll(__ballot(L.s[s] < x));
  if (pos >= 64 * M) return;
  uint64_t carry = x;  // last key of the previous slot (x before slot 0)
#pragma unroll
  for (int s = 0; s < M; ++s) {
    const uint64_t v = L.s[s];
    const uint64_t up = bperm64(v, lane == 0 ? 0 : lane - 1);
    const int e = s * 64 + lane;
    const uint64_t prev = lane == 0 ? carry : up;
    const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)v, 63);
    const uint32_t hi = __builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), 63);
    carry = ((uint64_t)hi << 32) | lo;
    L.s[s] = e < pos ? v : (e == pos ? x : prev);
  }
}

// Largest squared distance from qp to the k points of a previous result row
// (hint_pts by id), or -1 when the row is not k distinct points of the
// instance [lo, hi) other than the query itself.  Any k such points bound the
// query's k-th squared distance from above.
template <int M>
__device__ __forceinline__ float hint_bound(const QueryArgs& a, int out_row, const float4& qp, int self, int lo,
                                            int hi, int lane) {
  float mx = 0.f;
  bool bad = false;
#pragma unroll
  for (int s = 0; s < M; ++s) {
    const int j = s * 64 + lane;
    if (j < a.k) {
      const int id = a.out[(long long)out_row * a.k + j];
      if (id < lo || id >= hi || id == self)
        bad = true;
      else
        mx = fmaxf(mx, dist2(a.hint_pts[id], qp));
    }
  }
  if (__ballot(bad) != 0) return -1.f;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
  return mx;
}

// Squared distance from q to the box of cell (cx,cy,cz), minus the slack,
// scaled down so that any point binned in that cell has a larger FP32 d2.
__device__ __forceinline__ float cell_bound(const GridShape& g, const float4& q, int cx, int cy, int cz) {
  const int c[3] = {cx, cy, cz};
  const float qq[3] = {q.x, q.y, q.z};
  float s = 0.f;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float lo = g.lo[a] + (float)c[a] * g.h;
    const float hi = lo + g.h;
    float d = 0.f;
    if (qq[a] < lo) d = lo - qq[a];
    if (qq[a] > hi) d = qq[a] - hi;
    d = fmaxf(0.f, d - g.slack);
    s = fmaf(d, d, s);
  }
  return s * (1.f - 1e-5f);
}

// Waves per workgroup of the query kernel: 2, 4 or 8 (knn_query's `waves`);
// each wave works alone, the workgroup size only changes how waves share a
// CU's LDS and are scheduled.
constexpr int kQueryWavesDefault = 4;

// Consecutive queries (tets of one region, or sites of one grid cell) are
// close to each other: a wave takes a run of kQueryRun of them, and each
// query starts from the previous one's k-th distance r and their distance d:
// the previous query's k neighbours lie within r + d of it (with itself in
// place of one that it excludes, mode 0 and 3), so its k-th key is below that
// bound (rounded up by a 1e-5 margin) and candidates beyond it are never
// staged, and the cell walk stops there.
//
// Fewer queries than kQueryRun for every wave that the GPU holds at once
// (kQueryFill) are spread over all of them instead, down to one query per
// wave, which walks the grid alone (kNN phase at 10,368 tets / 1,037 sites:
// 115 us in runs of 6 or 5, 79 in runs of 2 and 1; 146,334 tets / 14,633
// sites: 275 us, 269; the same from 4,096 to 8,192).
#ifndef VD_KNN_RUN
#define VD_KNN_RUN 6
#endif
#ifndef VD_KNN_FILL
#define VD_KNN_FILL 4096
#endif
constexpr int kQueryRun = VD_KNN_RUN, kQueryFill = VD_KNN_FILL;

// After the first query of a run, the points that the run's other queries can
// need are gathered once into LDS (at most kUnionCap): query i's k-th distance
// is at most r0 + |q_i - q_0| (the first query's k neighbours, with q_0 in
// place of q_i itself where the query excludes itself), so every point such a
// query can keep lies within R = max_i(|q_i - c| + r0 + |q_i - q_0|) of the
// centre c of the run.  Those queries scan the list instead of walking the
// grid, with the same keys and the same bounds, so their results are the
// same; a run whose list would not fit walks as before.
//
// What bounds the kernel is the issue of vector instructions, with 4 waves per
// SIMD not quite: at 5 the list is held to the LDS of a fifth of a CU (lists of
// tet queries, M = 1, take some 110 points, of site queries, M = 2, some 350)
// and the registers to a fifth of a SIMD's.  kNN phase at 1M tets / 100,000
// sites 1.55 -> 1.42 ms, 100,000 points and 1M random queries 2.14 -> 1.99 (M =
// 1 with 192 or 320 points 1.44, M = 2 with 320 points 1.43, with 448 and 4
// waves 1.49; 6 waves, whose registers spill more than the 12 and 20 that they
// do at 5, 1.98).  Past k = 128 the list is longer, at the 4 waves that its
// registers and LDS allow (the bound asks for 3).
template <int M>
struct QueryShape {
  static constexpr int kUnionCap = M == 1 ? 256 : M == 2 ? 384 : 512;
  static constexpr int kWavesPerSimd = M <= 2 ? 5 : 3;
};

// At most this many keys staged after the last merge are inserted one at a
// time instead of sorted and merged.
#ifndef VD_KNN_INSERT_MAX
#define VD_KNN_INSERT_MAX 6
#endif
constexpr int kInsertMax = VD_KNN_INSERT_MAX;

// Point of query q, its excluded reference id (or -1), output row and instance.
__device__ __forceinline__ void query_point(const QueryArgs& a, int q, float4& qp, int& self, int& out_row, int& inst) {
  self = -1;
  out_row = q;
  inst = 0;
  if (a.mode == 0) {
    qp = a.sorted_pts[q];
    self = a.sorted_ids[q];
    out_row = self;
    if (a.pt_inst) inst = a.pt_inst[self];
  } else if (a.mode == 3) {
    self = a.q_ids[q];
    qp = a.qpts[self];
    if (a.pt_inst) inst = a.pt_inst[self];
  } else {
    if (a.q_inst) inst = a.q_inst[q];
    if (a.mode == 1) {
      const int4 t = a.tets[q];
      const float4 v0 = a.verts[t.x], v1 = a.verts[t.y], v2 = a.verts[t.z], v3 = a.verts[t.w];
      qp.x = (((v0.x + v1.x) + v2.x) + v3.x) * 0.25f;
      qp.y = (((v0.y + v1.y) + v2.y) + v3.y) * 0.25f;
      qp.z = (((v0.z + v1.z) + v2.z) + v3.z) * 0.25f;
      qp.w = 0.f;
    } else {
      qp = a.qpts[q];
    }
  }
}

template <int M, int kQueryWaves>
__global__ __launch_bounds__(64 * kQueryWaves, QueryShape<M>::kWavesPerSimd) void k_knn_query(QueryArgs a) {
  constexpr int kUnionCap = QueryShape<M>::kUnionCap;
  __shared__ uint64_t stage_all[kQueryWaves][128];
  __shared__ int mark_all[kQueryWaves][64];  // batch_owner's marks
  __shared__ float4 uni_all[kQueryWaves][kUnionCap];  // (x, y, z, id bits)
  const int lane = threadIdx.x & 63;
  const int wv = threadIdx.x >> 6;
  uint64_t* stage = stage_all[wv];
  int* mark = mark_all[wv];
  float4* uni = uni_all[wv];
  const int run = a.run;
  const int q0 = (blockIdx.x * kQueryWaves + wv) * run;
  int nq = a.n_query;
  if (a.n_query_dev) nq = min(nq, (int)min(*a.n_query_dev, (unsigned)a.n_query));
  float prev_r = -1.f;
  float4 prev_qp = {0.f, 0.f, 0.f, 0.f};
  int prev_inst = -1;
  // the run's point list: n_uni points (-1: none), valid for instance uni_inst
  int n_uni = -1, uni_inst = -1;
  float r0 = 0.f;
  float4 q0p = {0.f, 0.f, 0.f, 0.f};
  // with previous results (hint_pts): lane j holds the hint bound of query
  // q0 + j once it is known (-2 before; -1: that row gives none)
  const bool use_hint = a.hint_pts && a.out_pitch <= 0 && (a.mode == 0 || a.mode == 1);
  float run_hb = -2.f;
  // Results by columns (pitched, one column per query) that wait to be written
  // together: n_held queries from q_held on, in the space of the point list
  // while there is none.  A row of such a result has the run's queries side by
  // side, and one store then covers ten rows instead of 64.
  const bool hold = a.out_pitch > 0 && (a.mode == 1 || a.mode == 2) && run > 1;
  int* held = (int*)uni;  // [n_held][a.k + 1]
  static_assert(kQueryRun * (64 * M + 1) * sizeof(int) <= kUnionCap * sizeof(float4), "held results");
  int n_held = 0, q_held = q0;
  auto write_held = [&]() {
    if (n_held == 0) return;
    wave_sync();
    const int rows = 64 / n_held, j0 = lane / n_held, i = lane - j0 * n_held;
    if (j0 < rows)
      for (int j = j0; j < a.k; j += rows) a.out[(long long)j * a.out_pitch + q_held + i] = held[i * (a.k + 1) + j];
    wave_sync();
    n_held = 0;
  };
  // The run's point list: every point of the instance within sqrt(R2) of c,
  // with its id in w; returns their number, or -1 when they do not fit in
  // kUnionCap or the offset table does not reach that far (beyond it the
  // walk scans the whole instance: no list).
  auto gather = [&](const float4& c, float R2, const GridShape& g, int cbase) -> int {
    const int cc[3] = {cell_coord(c.x, g.lo[0], g.inv_h, g.dim[0]), cell_coord(c.y, g.lo[1], g.inv_h, g.dim[1]),
                       cell_coord(c.z, g.lo[2], g.inv_h, g.dim[2])};
    int n = 0;
    bool fits = true, covered = false;
    for (int ob = 0; ob < a.n_offsets && fits; ob += 64) {
      const float lbd = fmaxf(0.f, sqrtf((float)a.offsets[ob].w) * g.h - 2.f * g.slack);
      if (lbd * lbd * (1.f - 1e-5f) > R2) {
        covered = true;  // offsets are sorted by lb: the rest are beyond R too
        break;
      }
      int cnt = 0, st = 0;
      const int oi = ob + lane;
      if (oi < a.n_offsets) {
        const int4 o = a.offsets[oi];
        const int ox = cc[0] + o.x, oy = cc[1] + o.y, oz = cc[2] + o.z;
        if (ox >= 0 && ox < g.dim[0] && oy >= 0 && oy < g.dim[1] && oz >= 0 && oz < g.dim[2] &&
            !(cell_bound(g, c, ox, oy, oz) > R2)) {
          const int cell = cbase + ox + g.dim[0] * (oy + g.dim[1] * oz);
          st = a.start[cell];
          cnt = a.start[cell + 1] - st;
        }
      }
      const int incl = wave_incl_sum(cnt);
      const int excl = incl - cnt;
      const int total = __shfl(incl, 63);
      int carry = 0;
      for (int f0 = 0; f0 < total && fits; f0 += 64) {
        const int f = f0 + lane;
        const int own = batch_owner(mark, lane, cnt, excl, f0, carry);
        const int o_st = __shfl(st, own), o_ex = __shfl(excl, own);
        bool keep = false;
        float4 p = {0.f, 0.f, 0.f, 0.f};
        if (f < total) {
          const int idx = o_st + (f - o_ex);
          p = a.sorted_pts[idx];
          keep = !(dist2(p, c) > R2);
        }
        const uint64_t m = __ballot(keep);
        const int below = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
        const int add = __popcll(m);
        if (n + add > kUnionCap) {
          fits = false;
        } else {
          if (keep) uni[n + below] = p;
          n += add;
        }
      }
    }
    if (!(fits && covered)) return -1;
    wave_sync();
    return n;
  };
  // With previous results (hint_pts) every query of the run has a bound on its
  // k-th distance before any walk: the run's list is then gathered first,
  // within max_j(|q_j - c| + r_j) of the centre c of the run's queries (r_j:
  // query j's bound), and every query of the run, the first one included,
  // scans it instead of walking the grid, with the walk's keys and bounds.
  if (use_hint && run > 1) {
    const int n_run = min(q0 + run, nq) - q0;
    float4 pj = {0.f, 0.f, 0.f, 0.f};
    int sj = -1, rj = 0, ij = 0;
    const bool in = lane < n_run;
    if (in) query_point(a, q0 + lane, pj, sj, rj, ij);
    const int inst0 = __shfl(ij, 0);
    if (n_run > 0 && __ballot(in && ij != inst0) == 0) {
      const int lo = a.pt_begin ? a.pt_begin[inst0] : 0, hi = a.pt_begin ? a.pt_begin[inst0 + 1] : a.n_ref;
      for (int j = 0; j < n_run; ++j) {
        const float4 qj4 = make_float4(__shfl(pj.x, j), __shfl(pj.y, j), __shfl(pj.z, j), 0.f);
        const float hb = hint_bound<M>(a, __shfl(rj, j), qj4, __shfl(sj, j), lo, hi, lane);
        if (lane == j) run_hb = hb;
      }
      if (__ballot(in && !(run_hb >= 0.f)) == 0) {
        float cx = in ? pj.x : 0.f, cy = in ? pj.y : 0.f, cz = in ? pj.z : 0.f;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
          cx += __shfl_xor(cx, o);
          cy += __shfl_xor(cy, o);
          cz += __shfl_xor(cz, o);
        }
        const float inv = 1.f / (float)n_run;
        const float4 c = make_float4(cx * inv, cy * inv, cz * inv, 0.f);
        float need = 0.f;
        if (in) {
          const float ax = pj.x - c.x, ay = pj.y - c.y, az = pj.z - c.z;
          need = sqrtf(fmaf(az, az, fmaf(ay, ay, ax * ax))) + sqrtf(run_hb);
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) need = fmaxf(need, __shfl_xor(need, o));
        const GridShape g = a.grid[inst0];
        // rounding margins of the FP32 distances on either side
        const float R = need * (1.f + 1e-4f) + 1e-3f * g.h;
        const int n = gather(c, R * R, g, a.cell_base ? a.cell_base[inst0] : 0);
        if (n >= 0) {
          n_uni = n;
          uni_inst = inst0;
          r0 = INFINITY;  // the queries' own bounds hold
        }
      }
    }
  }
  for (int q = q0; q < q0 + run && q < nq; ++q) {  // wave-uniform

  float4 qp;
  int self, out_row, inst;
  query_point(a, q, qp, self, out_row, inst);
  const GridShape g = a.grid[inst];
  const int cbase = a.cell_base ? a.cell_base[inst] : 0;
  const bool from_list = n_uni >= 0 && inst == uni_inst;
  const int qc[3] = {cell_coord(qp.x, g.lo[0], g.inv_h, g.dim[0]), cell_coord(qp.y, g.lo[1], g.inv_h, g.dim[1]),
                     cell_coord(qp.z, g.lo[2], g.inv_h, g.dim[2])};

  TopK<M> L;
#pragma unroll
  for (int s = 0; s < M; ++s) L.s[s] = kNoKey;
  uint64_t bound = kNoKey;
  if (prev_r >= 0.f && prev_inst == inst) {
    const float dx = qp.x - prev_qp.x, dy = qp.y - prev_qp.y, dz = qp.z - prev_qp.z;
    const float b = prev_r + sqrtf(fmaf(dz, dz, fmaf(dy, dy, dx * dx)));
    const float b2 = b * b * (1.f + 1e-5f);
    if (b2 < INFINITY) bound = key_bound(b2);
  }
  if (from_list) {
    // the bound the list was gathered for: r0 + |q - q0|
    const float dx = qp.x - q0p.x, dy = qp.y - q0p.y, dz = qp.z - q0p.z;
    const float b = r0 + sqrtf(fmaf(dz, dz, fmaf(dy, dy, dx * dx)));
    const float b2 = b * b * (1.f + 1e-5f);
    bound = umin64(bound, key_bound(b2));
  }
  if (use_hint) {
    // the query's previous result: its k points' current distances
    float hb = __shfl(run_hb, q - q0);
    if (hb == -2.f) {
      const int lo = a.pt_begin ? a.pt_begin[inst] : 0, hi = a.pt_begin ? a.pt_begin[inst + 1] : a.n_ref;
      hb = hint_bound<M>(a, out_row, qp, self, lo, hi, lane);
    }
    if (hb >= 0.f) bound = umin64(bound, key_bound(hb));
  }
  uint64_t thr = bound;
  int staged = 0;
  bool done = false;
  bool empty = true;  // no key merged yet (wave-uniform)

  auto push = [&](uint64_t key, bool ok) {
    const uint64_t mask = __ballot(ok);
    const int below = __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0));
    if (ok) stage[staged + below] = key;
    staged += __popcll(mask);
    wave_sync();
    if (staged >= 64) {
      const uint64_t x = stage[lane];
      const uint64_t rest = (lane + 64 < staged) ? stage[lane + 64] : kNoKey;
      wave_sync();
      if (lane + 64 < staged) stage[lane] = rest;
      staged -= 64;
      wave_sync();
      topk_merge<M>(L, x, lane, empty);
      empty = false;
      thr = umin64(bound, topk_kth<M>(L, a.k));
    }
  };

  if (from_list) {
    for (int f0 = 0; f0 < n_uni; f0 += 64) {
      const int f = f0 + lane;
      uint64_t key = kNoKey;
      bool ok = false;
      if (f < n_uni) {
        const float4 p = uni[f];
        const uint32_t id = __float_as_uint(p.w);
        key = knn_key(dist2(p, qp), id);
        ok = ((int)id != self) && key < thr;
      }
      push(key, ok);
    }
    done = true;
  }
  for (int ob = 0; ob < a.n_offsets && !done; ob += 64) {
    const float kth = key_d2(thr);
    // offsets are sorted by lb: once the first of the batch is beyond the k-th
    // distance, so are all later ones
    const float lbd = fmaxf(0.f, sqrtf((float)a.offsets[ob].w) * g.h - 2.f * g.slack);
    if (thr != kNoKey && lbd * lbd * (1.f - 1e-5f) > kth) {
      done = true;
      break;
    }
    int cnt = 0, st = 0;
    const int oi = ob + lane;
    if (oi < a.n_offsets) {
      const int4 o = a.offsets[oi];
      const int cx = qc[0] + o.x, cy = qc[1] + o.y, cz = qc[2] + o.z;
      if (cx >= 0 && cx < g.dim[0] && cy >= 0 && cy < g.dim[1] && cz >= 0 && cz < g.dim[2]) {
        if (thr == kNoKey || !(cell_bound(g, qp, cx, cy, cz) > kth)) {
          const int c = cbase + cx + g.dim[0] * (cy + g.dim[1] * cz);
          st = a.start[c];
          cnt = a.start[c + 1] - st;
        }
      }
    }
    // exclusive prefix of the counts across the wave
    const int incl = wave_incl_sum(cnt);
    const int excl = incl - cnt;
    const int total = __shfl(incl, 63);
    int carry = 0;
    for (int f0 = 0; f0 < total; f0 += 64) {
      const int f = f0 + lane;
      const int own = batch_owner(mark, lane, cnt, excl, f0, carry);
      const int o_st = __shfl(st, own), o_ex = __shfl(excl, own);
      uint64_t key = kNoKey;
      bool ok = false;
      if (f < total) {
        const int idx = o_st + (f - o_ex);
        const float4 p = a.sorted_pts[idx];
        const int id = __float_as_int(p.w);
        key = knn_key(dist2(p, qp), (uint32_t)id);
        ok = (id != self) && key < thr;
      }
      push(key, ok);
    }
  }
  if (!done) {
    // offsets table exhausted without the stop test passing: scan all points
    // of the instance
    const int r0 = a.start[cbase], r1 = a.start[cbase + g.ncell];
    for (int f0 = r0; f0 < r1; f0 += 64) {
      const int f = f0 + lane;
      uint64_t key = kNoKey;
      bool ok = false;
      if (f < r1) {
        // skip cells already visited: those inside the offset table's reach
        const float4 p = a.sorted_pts[f];
        const int id = __float_as_int(p.w);
        const int cx = cell_coord(p.x, g.lo[0], g.inv_h, g.dim[0]) - qc[0];
        const int cy = cell_coord(p.y, g.lo[1], g.inv_h, g.dim[1]) - qc[1];
        const int cz = cell_coord(p.z, g.lo[2], g.inv_h, g.dim[2]) - qc[2];
        const int r = max(abs(cx), max(abs(cy), abs(cz)));
        key = knn_key(dist2(p, qp), (uint32_t)id);
        ok = (r > kOffsetRadius) && (id != self) && key < thr;
      }
      push(key, ok);
    }
  }
  if (staged > 0 && !empty && staged <= kInsertMax) {
    // a few keys past the last merge: inserted one by one
    for (int i = 0; i < staged; ++i) {
      const uint64_t x = stage[i];
      if (x < thr) {
        topk_insert<M>(L, x, lane);
        thr = umin64(bound, topk_kth<M>(L, a.k));
      }
    }
  } else if (staged > 0) {
    const uint64_t x = lane < staged ? stage[lane] : kNoKey;
    topk_merge<M>(L, x, lane, empty);
  }
#pragma unroll
  for (int s = 0; s < M; ++s) {
    const int j = s * 64 + lane;
    if (j < a.k) {
      const int32_t id = L.s[s] == kNoKey ? -1 : (int32_t)(uint32_t)L.s[s];
      if (hold && n_uni < 0)
        held[(q - q_held) * (a.k + 1) + j] = id;
      else if (a.out_pitch > 0)
        a.out[(long long)j * a.out_pitch + out_row] = id;
      else
        a.out[(long long)out_row * a.k + j] = id;
    }
  }
  if (hold && n_uni < 0)
    ++n_held;
  else
    q_held = q + 1;
  const uint64_t kth = topk_kth<M>(L, a.k);
  prev_r = kth == kNoKey ? -1.f : sqrtf(key_d2(kth));
  prev_qp = qp;
  prev_inst = inst;

  const int q_end = min(q0 + run, nq);
  if (q == q0 && n_uni < 0 && prev_r >= 0.f && q + 1 < q_end) {
    // the run's other queries: their points (lane j takes query q0 + j)
    float4 pj = qp;
    int sj = self, rj = out_row, ij = inst;
    const int qj = q0 + lane;
    if (lane >= 1 && qj < q_end) query_point(a, qj, pj, sj, rj, ij);
    const bool in = lane >= 1 && qj < q_end;
    const bool same = __ballot(in && ij != inst) == 0;
    if (same) {
      const int n_in = q_end - q0 - 1;
      float cx = in ? pj.x : 0.f, cy = in ? pj.y : 0.f, cz = in ? pj.z : 0.f;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        cx += __shfl_xor(cx, o);
        cy += __shfl_xor(cy, o);
        cz += __shfl_xor(cz, o);
      }
      const float inv = 1.f / (float)n_in;
      const float4 c = make_float4(cx * inv, cy * inv, cz * inv, 0.f);
      if (use_hint) {
        // the other queries' bounds from their previous results (lane j: query q0 + j)
        const int lo = a.pt_begin ? a.pt_begin[inst] : 0, hi = a.pt_begin ? a.pt_begin[inst + 1] : a.n_ref;
        for (int j = 1; j <= n_in; ++j) {
          const float4 qj4 = make_float4(__shfl(pj.x, j), __shfl(pj.y, j), __shfl(pj.z, j), 0.f);
          const int sj_row = __shfl(rj, j), sj_self = __shfl(sj, j);
          const float hb = hint_bound<M>(a, sj_row, qj4, sj_self, lo, hi, lane);
          if (lane == j) run_hb = hb;
        }
      }
      float rj_need = 0.f;
      if (in) {
        const float ax = pj.x - c.x, ay = pj.y - c.y, az = pj.z - c.z;
        const float bx = pj.x - qp.x, by = pj.y - qp.y, bz = pj.z - qp.z;
        float rq = prev_r + sqrtf(fmaf(bz, bz, fmaf(by, by, bx * bx)));
        if (run_hb >= 0.f) rq = fminf(rq, sqrtf(run_hb));
        rj_need = sqrtf(fmaf(az, az, fmaf(ay, ay, ax * ax))) + rq;
      }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) rj_need = fmaxf(rj_need, __shfl_xor(rj_need, o));
      // rounding margins of the FP32 distances on either side
      const float R = rj_need * (1.f + 1e-4f) + 1e-3f * g.h;
      const float R2 = R * R;
      // A ball of radius R as densely filled as the first query's holds
      // k (R / r0)^3 points; a gather of far more than the list takes (queries
      // in no spatial order) would fail after reading most of them: 100,000
      // points, 1M random queries 2.45 -> 2.24 ms, and 2.13 with the results held as above.
      const float rel = R / prev_r;
      if (!((float)a.k * rel * rel * rel > 2.f * (float)kUnionCap && prev_r > 0.f)) {
        write_held();  // the list takes their space
        q_held = q + 1;
        const int n = gather(c, R2, g, cbase);
        if (n >= 0) {
          n_uni = n;
          uni_inst = inst;
          r0 = prev_r;
          q0p = qp;
        }
      }
    }
  }
  }  // query loop
  write_held();
}

}  // namespace

__global__ void k_fill_u32(uint32_t* p, long long n, uint32_t v) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    p[i] = v;
}

hipError_t fill_u32(void* p, long long n, uint32_t v, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  const long long blocks = std::min<long long>((n + 255) / 256, 4096);
  hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)blocks), dim3(256), 0, st, (uint32_t*)p, n, v);
  return hipGetLastError();
}

__global__ void k_clear(ClearList l) {
  for (int i = 0; i < l.n; ++i)
    for (long long j = (long long)blockIdx.x * blockDim.x + threadIdx.x; j < l.words[i];
         j += (long long)gridDim.x * blockDim.x)
      l.p[i][j] = 0u;
}

hipError_t clear_all(const ClearList& l, hipStream_t st) {
  long long most = 0;
  for (int i = 0; i < l.n; ++i) most = std::max(most, l.words[i]);
  if (most <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_clear, dim3((unsigned)std::min<long long>((most + 255) / 256, 4096)), dim3(256), 0, st, l);
  return hipGetLastError();
}

// Exclusive scan, three passes: per-block scans of kScanTile items, a scan of
// the block totals, then the block offsets added back.  Also clears `cursor`.
constexpr int kScanItems = 8;
constexpr int kScanTile = 1024 * kScanItems;

__device__ __forceinline__ int scan_n(const int* n_dev, int n_max) { return n_dev ? min(*n_dev, n_max) : n_max; }

// T: int, or unsigned for totals up to 2^32 - 1.
template <class T>
__global__ __launch_bounds__(1024) void k_scan_tiles(const int* in, const int* n_dev, int n_max, T* out,
                                                      int* cursor, T* tile_sum) {
  __shared__ T part[1024];
  const int n = scan_n(n_dev, n_max);
  const long long base = (long long)blockIdx.x * kScanTile;
  if (base >= n && blockIdx.x > 0) return;
  const bool only = n_max <= kScanTile;  // the tile is the whole scan
  T v[kScanItems];
  T s = 0;
#pragma unroll
  for (int j = 0; j < kScanItems; ++j) {
    const long long i = base + (long long)j * 1024 + threadIdx.x;
    v[j] = i < n ? (T)in[i] : (T)0;
  }
  // thread t owns items base + t*kScanItems .. ; reorder through LDS for that
  __shared__ T tile[kScanTile];
#pragma unroll
  for (int j = 0; j < kScanItems; ++j) tile[j * 1024 + threadIdx.x] = v[j];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kScanItems; ++j) {
    v[j] = tile[threadIdx.x * kScanItems + j];
    s += v[j];
  }
  part[threadIdx.x] = s;
  __syncthreads();
  for (int off = 1; off < 1024; off <<= 1) {
    const T x = threadIdx.x >= off ? part[threadIdx.x - off] : (T)0;
    __syncthreads();
    part[threadIdx.x] += x;
    __syncthreads();
  }
  T run = part[threadIdx.x] - s;
#pragma unroll
  for (int j = 0; j < kScanItems; ++j) {
    tile[threadIdx.x * kScanItems + j] = run;
    run += v[j];
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kScanItems; ++j) {
    const long long i = base + (long long)j * 1024 + threadIdx.x;
    if (i < n) {
      out[i] = tile[j * 1024 + threadIdx.x];
      if (cursor) cursor[i] = 0;
    }
  }
  if (threadIdx.x == 1023) {
    if (only)
      out[n] = part[1023];
    else
      tile_sum[blockIdx.x] = part[1023];
  }
}

template <class T>
__global__ __launch_bounds__(1024) void k_scan_top(const int* n_dev, int n_max, T* tile_sum) {
  __shared__ T part[1024];
  const int n = scan_n(n_dev, n_max);
  const int tiles = (n + kScanTile - 1) / kScanTile;
  const int per = (tiles + 1023) / 1024;
  const int b = threadIdx.x * per, e = min(tiles, b + per);
  T s = 0;
  for (int i = b; i < e; ++i) s += tile_sum[i];
  part[threadIdx.x] = s;
  __syncthreads();
  for (int off = 1; off < 1024; off <<= 1) {
    const T x = threadIdx.x >= off ? part[threadIdx.x - off] : (T)0;
    __syncthreads();
    part[threadIdx.x] += x;
    __syncthreads();
  }
  T run = part[threadIdx.x] - s;
  for (int i = b; i < e; ++i) {
    const T t = tile_sum[i];
    tile_sum[i] = run;
    run += t;
  }
  if (threadIdx.x == 1023) tile_sum[tiles] = part[1023];
}

template <class T>
__global__ void k_scan_add(const int* n_dev, int n_max, T* out, const T* tile_sum) {
  const int n = scan_n(n_dev, n_max);
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] += tile_sum[i / kScanTile];
  if (i == n) out[n] = tile_sum[(n + kScanTile - 1) / kScanTile];
}

int scan_tmp_ints(int n_max) { return (n_max + kScanTile - 1) / kScanTile + 2; }

template <class T>
static hipError_t scan_excl_t(const int* in, const int* n_dev, int n_max, T* out, int* cursor, T* tmp,
                              hipStream_t st) {
  const int tiles = std::max(1, (n_max + kScanTile - 1) / kScanTile);
  hipLaunchKernelGGL(k_scan_tiles<T>, dim3(tiles), dim3(1024), 0, st, in, n_dev, n_max, out, cursor, tmp);
  if (n_max <= kScanTile) return hipGetLastError();
  hipLaunchKernelGGL(k_scan_top<T>, dim3(1), dim3(1024), 0, st, n_dev, n_max, tmp);
  hipLaunchKernelGGL(k_scan_add<T>, dim3((unsigned)(((long long)n_max + 1 + 255) / 256)), dim3(256), 0, st, n_dev,
                     n_max, out, tmp);
  return hipGetLastError();
}
hipError_t scan_excl(const int* in, const int* n_dev, int n_max, int* out, int* cursor, int* tmp, hipStream_t st) {
  return scan_excl_t<int>(in, n_dev, n_max, out, cursor, tmp, st);
}
hipError_t scan_excl(const int* in, const int* n_dev, int n_max, unsigned* out, int* cursor, unsigned* tmp,
                     hipStream_t st) {
  return scan_excl_t<unsigned>(in, n_dev, n_max, out, cursor, tmp, st);
}

static std::vector<int4> make_offset_table() {
  std::vector<int4> t;
  const int R = kOffsetRadius;
  for (int z = -R; z <= R; ++z)
    for (int y = -R; y <= R; ++y)
      for (int x = -R; x <= R; ++x) {
        auto m = [](int d) { return std::max(std::abs(d) - 1, 0); };
        t.push_back(make_int4(x, y, z, m(x) * m(x) + m(y) * m(y) + m(z) * m(z)));
      }
  std::stable_sort(t.begin(), t.end(), [](const int4& a, const int4& b) {
    if (a.w != b.w) return a.w < b.w;
    const int ca = std::max(std::abs(a.x), std::max(std::abs(a.y), std::abs(a.z)));
    const int cb = std::max(std::abs(b.x), std::max(std::abs(b.y), std::abs(b.z)));
    return ca < cb;
  });
  return t;
}
const std::vector<int4>& knn_offset_table() {
  static const std::vector<int4> t = make_offset_table();
  return t;
}

int grid_max_cells(int n, float density) {
  const double c = std::max(1.0, n / (double)density);
  return (int)std::min(64.0 * 1024 * 1024, std::max(64.0, 1.25 * c + 64.0));
}

hipError_t grid_build(const GridBufs& gb, const float4* pts, int n, const float* extra_lo, const float* extra_hi,
                      float density, hipStream_t st) {
  const float3 elo = extra_lo ? make_float3(extra_lo[0], extra_lo[1], extra_lo[2]) : make_float3(0, 0, 0);
  const float3 ehi = extra_hi ? make_float3(extra_hi[0], extra_hi[1], extra_hi[2]) : make_float3(0, 0, 0);
  if (gb.n_inst < 1 || (gb.n_inst > 1 && (!gb.cell_base || !gb.pt_begin || !gb.pt_inst))) return hipErrorInvalidValue;
  const int max_pts = gb.n_inst == 1 ? n : gb.max_pts;
  if (max_pts > 0 && max_pts <= kSmallPoints &&
      (gb.n_inst == 1 ? gb.max_cells : grid_max_cells(max_pts, density)) <= kSmallCells) {
    hipLaunchKernelGGL(k_grid_small, dim3((unsigned)gb.n_inst), dim3(kScanThreads), 0, st, pts, n, gb.pt_begin,
                       gb.cell_base, gb.box, elo, ehi, extra_lo ? 1 : 0, density, gb.max_cells, gb.n_inst, gb.shape,
                       gb.count, gb.start, gb.sorted_ids, gb.sorted_pts);
    return hipGetLastError();
  }
  // the parts' boxes in the count table, which is cleared after the shape
  const bool parts = gb.n_inst == 1 && !gb.pt_begin && n > kSmallPoints && gb.max_cells >= 6 * kBoxParts;
  if (parts)
    hipLaunchKernelGGL(k_grid_box, dim3(kBoxParts), dim3(kScanThreads), 0, st, pts, n, (float*)gb.count);
  hipLaunchKernelGGL(k_grid_shape, dim3((unsigned)gb.n_inst), dim3(parts ? 64 : kScanThreads), 0, st, pts, n,
                     gb.pt_begin, gb.cell_base, gb.box, elo, ehi, extra_lo ? 1 : 0, density, gb.max_cells,
                     parts ? (const float*)gb.count : nullptr, kBoxParts, gb.shape);
  hipError_t e = fill_u32(gb.count, gb.max_cells, 0u, st);
  if (e != hipSuccess) return e;
  const int nb = (n + 255) / 256;
  if (n > 0)
    hipLaunchKernelGGL(k_grid_count, dim3(nb), dim3(256), 0, st, pts, n, gb.shape, gb.pt_inst, gb.cell_base,
                       gb.cell_of, gb.count);
  // one instance: scan only the cells in use; a batch: all cells (unused
  // ones are empty)
  e = scan_excl(gb.count, gb.n_inst == 1 ? &gb.shape->ncell : nullptr, gb.max_cells, gb.start, gb.cursor,
                gb.scan_tmp, st);
  if (e != hipSuccess) return e;
  if (n > 0)
    hipLaunchKernelGGL(k_grid_scatter, dim3(nb), dim3(256), 0, st, n, gb.cell_of, gb.start, gb.cursor,
                       gb.sorted_ids);
  hipLaunchKernelGGL(k_grid_sort, dim3((gb.max_cells + kSortCells - 1) / kSortCells), dim3(kSortThreads), 0, st,
                     gb.shape, gb.n_inst == 1 ? -1 : gb.max_cells, pts, gb.start, gb.sorted_ids, gb.sorted_pts);
  return hipGetLastError();
}

namespace {
template <int W>
hipError_t launch_query_w(const QueryArgs& a, int n_query, hipStream_t st) {
  const dim3 grid((n_query + W * a.run - 1) / (W * a.run)), block(64 * W);
  if (a.k <= 64)
    hipLaunchKernelGGL((k_knn_query<1, W>), grid, block, 0, st, a);
  else if (a.k <= 128)
    hipLaunchKernelGGL((k_knn_query<2, W>), grid, block, 0, st, a);
  else
    hipLaunchKernelGGL((k_knn_query<4, W>), grid, block, 0, st, a);
  return hipGetLastError();
}
hipError_t launch_query(QueryArgs a, int n_query, int waves, hipStream_t st) {
  a.run = std::max(1, std::min(kQueryRun, n_query / kQueryFill));
  if (waves == 2) return launch_query_w<2>(a, n_query, st);
  if (waves == 8) return launch_query_w<8>(a, n_query, st);
  return launch_query_w<kQueryWavesDefault>(a, n_query, st);
}
}  // namespace

hipError_t knn_query(const GridBufs& gb, int n_ref, const int4* offsets, int n_offsets, int k, int mode,
                     int n_query, const float4* verts, const int4* tets, const float4* qpts, const int* q_inst,
                     int32_t* out, long long out_pitch, hipStream_t st, const float4* hint_pts, int waves) {
  if (k < 1 || k > 256) return hipErrorInvalidValue;
  QueryArgs a;
  a.hint_pts = hint_pts;
  a.pt_begin = gb.pt_begin;
  a.grid = gb.shape;
  a.cell_base = gb.cell_base;
  a.pt_inst = gb.pt_inst;
  a.q_inst = q_inst;
  a.sorted_pts = gb.sorted_pts;
  a.sorted_ids = gb.sorted_ids;
  a.start = gb.start;
  a.n_ref = n_ref;
  a.offsets = offsets;
  a.n_offsets = n_offsets;
  a.k = k;
  a.n_query = n_query;
  a.mode = mode;
  a.verts = verts;
  a.tets = tets;
  a.qpts = qpts;
  a.out = out;
  a.out_pitch = out_pitch;
  a.q_ids = nullptr;
  a.n_query_dev = nullptr;
  if (n_query <= 0) return hipSuccess;
  return launch_query(a, n_query, waves, st);
}

hipError_t knn_query_ids(const GridBufs& gb, const int4* offsets, int n_offsets, int k, const float4* pts,
                         const int* ids, const unsigned* n_ids_dev, int n_ids_max, int32_t* out, hipStream_t st) {
  if (k < 1 || k > 256) return hipErrorInvalidValue;
  if (n_ids_max <= 0) return hipSuccess;
  QueryArgs a;
  a.hint_pts = nullptr;
  a.pt_begin = gb.pt_begin;
  a.grid = gb.shape;
  a.cell_base = gb.cell_base;
  a.pt_inst = gb.pt_inst;
  a.q_inst = nullptr;
  a.sorted_pts = gb.sorted_pts;
  a.sorted_ids = gb.sorted_ids;
  a.start = gb.start;
  a.n_ref = 0;
  a.offsets = offsets;
  a.n_offsets = n_offsets;
  a.k = k;
  a.n_query = n_ids_max;
  a.mode = 3;
  a.verts = nullptr;
  a.tets = nullptr;
  a.qpts = pts;
  a.out = out;
  a.out_pitch = 0;
  a.q_ids = ids;
  a.n_query_dev = n_ids_dev;
  return launch_query(a, n_ids_max, kQueryWavesDefault, st);
}

}  // namespace vd
