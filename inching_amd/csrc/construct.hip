// Construction kernels for gfx950: cell-list neighbour search and ANM 3x3
// super-element assembly into full-storage block rows.
//
// Neighbour rule (shared with assembly and the matrix-free operator):
//   j in ball(i)  <=>  (dx*dx + dy*dy) + dz*dz <= rc*rc,  dx = x_j - x_i (float64),
// evaluated with explicit round-to-nearest operations so no FMA contraction can
// change the set.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>

#include "common.h"
#include "scan.h"
#include "tile.h"

#include <hipcub/hipcub.hpp>

namespace {

constexpr int kMaxRow = 2048;  // capacity of one neighbour row in the sort kernel

__device__ __forceinline__ double dist2(double dx, double dy, double dz) {
  return __dadd_rn(__dadd_rn(__dmul_rn(dx, dx), __dmul_rn(dy, dy)), __dmul_rn(dz, dz));
}

struct Grid {
  double lo[3];
  double inv;  // 1 / cell size
  int64_t dim[3];
};

__device__ __forceinline__ int64_t cell_coord(double v, double lo, double inv, int64_t dim) {
  int64_t c = (int64_t)floor((v - lo) * inv);
  return c < 0 ? 0 : (c >= dim ? dim - 1 : c);
}

// Minimum and maximum that propagate NaN (fmin/fmax drop it), so that a NaN coordinate
// reaches the host's finiteness check.
__device__ __forceinline__ double nan_min(double a, double b) { return (a < b || a != a) ? a : b; }
__device__ __forceinline__ double nan_max(double a, double b) { return (a > b || a != a) ? a : b; }

__global__ void k_minmax(int64_t n, const double *__restrict__ xyz, double *__restrict__ part) {
  // part[blockIdx.x*6 + {0..2}] = min, {3..5} = max; NaN in either when any coordinate is NaN
  __shared__ double smin[3][256], smax[3][256];
  double mn[3] = {INFINITY, INFINITY, INFINITY}, mx[3] = {-INFINITY, -INFINITY, -INFINITY};
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    for (int a = 0; a < 3; ++a) {
      double v = xyz[3 * i + a];
      mn[a] = nan_min(mn[a], v);
      mx[a] = nan_max(mx[a], v);
    }
  }
  for (int a = 0; a < 3; ++a) {
    smin[a][threadIdx.x] = mn[a];
    smax[a][threadIdx.x] = mx[a];
  }
  __syncthreads();
  for (int s = blockDim.x / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s)
      for (int a = 0; a < 3; ++a) {
        smin[a][threadIdx.x] = nan_min(smin[a][threadIdx.x], smin[a][threadIdx.x + s]);
        smax[a][threadIdx.x] = nan_max(smax[a][threadIdx.x], smax[a][threadIdx.x + s]);
      }
    __syncthreads();
  }
  if (threadIdx.x == 0)
    for (int a = 0; a < 3; ++a) {
      part[blockIdx.x * 6 + a] = smin[a][0];
      part[blockIdx.x * 6 + 3 + a] = smax[a][0];
    }
}

__global__ void k_cell_count(int64_t n, const double *__restrict__ xyz, Grid g, int32_t *__restrict__ cell_of,
                             int32_t *__restrict__ count) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  int64_t c[3];
  for (int a = 0; a < 3; ++a) c[a] = cell_coord(xyz[3 * i + a], g.lo[a], g.inv, g.dim[a]);
  int64_t id = (c[0] * g.dim[1] + c[1]) * g.dim[2] + c[2];
  cell_of[i] = (int32_t)id;
  atomicAdd(&count[id], 1);
}


__global__ void k_cell_fill(int64_t n, const int32_t *__restrict__ cell_of, const int32_t *__restrict__ start,
                            int32_t *__restrict__ cursor, int32_t *__restrict__ atoms) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  int32_t c = cell_of[i];
  int32_t p = atomicAdd(&cursor[c], 1);
  atoms[start[c] + p] = (int32_t)i;
}

// Coordinates in cell order.
__global__ void k_cell_coords(int64_t n, const double *__restrict__ xyz, const int32_t *__restrict__ atoms,
                              double *__restrict__ cx) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t >= 3 * n) return;
  cx[t] = xyz[3 * (int64_t)atoms[t / 3] + t % 3];
}

// A workgroup takes kRun atoms that are consecutive in cell order, column by column of cells (a
// run of one column needs the cells from one below its first to one above its last, in the
// nine columns around it: nine contiguous ranges of the cell order). The ranges' coordinates go
// through LDS, kStage at a time; a wave tests 64 of them at once against one of its atoms, and
// the lanes' ballot gives the count and each hit's place. Vector issue bounds it (busy in 72% and
// 67% of a CU's cycles, no bank conflicts): about 1,000 candidates an atom. One thread per atom, walking the 27 cells through memory, took 434 us per
// pass on 150,000 atoms; this takes 117 (counts) and 168 (columns).
// FILL = false: counts[i] and the longest row; FILL = true: the row's columns in cell order.
constexpr int kRun = 32, kStage = 1024;

template <bool FILL>
__global__ void __launch_bounds__(256) k_neigh(int64_t n, Grid g, double rc2, const int32_t *__restrict__ start,
                                               const int32_t *__restrict__ atoms, const double *__restrict__ cx,
                                               const int64_t *__restrict__ indptr, int64_t *__restrict__ counts,
                                               int32_t *__restrict__ longest, int32_t *__restrict__ indices) {
  __shared__ double sx[kStage], sy[kStage], sz[kStage];
  __shared__ int32_t sj[kStage];
  __shared__ double ax[kRun][3];
  __shared__ int64_t ac[kRun][3];
  __shared__ int32_t cnt[kRun], lo[9], hi[9];
  const int64_t t0 = blockIdx.x * (int64_t)kRun;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int na = (int)(n - t0 < kRun ? n - t0 : kRun);
  if (tid < na) {
    const double v[3] = {cx[3 * (t0 + tid)], cx[3 * (t0 + tid) + 1], cx[3 * (t0 + tid) + 2]};
    for (int a = 0; a < 3; ++a) {
      ax[tid][a] = v[a];
      ac[tid][a] = cell_coord(v[a], g.lo[a], g.inv, g.dim[a]);
    }
    cnt[tid] = 0;
  }
  __syncthreads();
  for (int r0 = 0; r0 < na;) {
    int r1 = r0 + 1;   // the run's atoms of one column: [r0, r1)
    while (r1 < na && ac[r1][0] == ac[r0][0] && ac[r1][1] == ac[r0][1]) ++r1;
    if (tid < 9) {
      const int64_t a = ac[r0][0] + tid / 3 - 1, b = ac[r0][1] + tid % 3 - 1;
      const bool in = a >= 0 && a < g.dim[0] && b >= 0 && b < g.dim[1];
      const int64_t c0 = ac[r0][2] > 0 ? ac[r0][2] - 1 : 0;
      const int64_t c1 = ac[r1 - 1][2] + 1 < g.dim[2] ? ac[r1 - 1][2] + 1 : g.dim[2] - 1;
      const int64_t id = (a * g.dim[1] + b) * g.dim[2];
      lo[tid] = in ? start[id + c0] : 0;
      hi[tid] = in ? start[id + c1 + 1] : 0;
    }
    __syncthreads();
    int total = 0;
#pragma unroll
    for (int k = 0; k < 9; ++k) total += hi[k] - lo[k];
    for (int base = 0; base < total; base += kStage) {
      const int m = total - base < kStage ? total - base : kStage;
      for (int q = tid; q < m; q += 256) {
        int p = base + q, k = 0;
        while (p >= hi[k] - lo[k]) {
          p -= hi[k] - lo[k];
          ++k;
        }
        p += lo[k];
        sx[q] = cx[3 * (int64_t)p];
        sy[q] = cx[3 * (int64_t)p + 1];
        sz[q] = cx[3 * (int64_t)p + 2];
        if (FILL) sj[q] = atoms[p];
      }
      __syncthreads();
      for (int r = r0 + w; r < r1; r += 4) {
        const double xi = ax[r][0], yi = ax[r][1], zi = ax[r][2];
        int c = cnt[r];
        int32_t *out = nullptr;
        int room = 0;
        if (FILL) {
          const int64_t i = atoms[t0 + r], b = indptr[i];
          out = indices + b;
          room = (int)(indptr[i + 1] - b);
        }
        for (int q0 = 0; q0 < m; q0 += 64) {
          const int q = q0 + lane;
          bool hit = false;
          if (q < m) hit = dist2(__dsub_rn(sx[q], xi), __dsub_rn(sy[q], yi), __dsub_rn(sz[q], zi)) <= rc2;
          const uint64_t bal = __ballot(hit);
          if (FILL && hit) {
            const int at = c + __popcll(bal & (((uint64_t)1 << lane) - 1));
            if (at < room) out[at] = sj[q];
          }
          c += __popcll(bal);
        }
        if (lane == 0) cnt[r] = c;
      }
      __syncthreads();
    }
    r0 = r1;
  }
  if (!FILL && tid < 64) {
    if (tid < na) counts[atoms[t0 + tid]] = cnt[tid];
    int m = tid < na ? cnt[tid] : 0;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const int o = __shfl_xor(m, off, 64);
      m = o > m ? o : m;
    }
    if (tid == 0 && m > *longest) atomicMax(longest, m);
  }
}

// Periodic images in x and y (membrane boxes): image s = (sx, sy) in {-1,0,1}^2 shifts atom j
// by (sx * bx, sy * by, 0); bit (sx + 1) * 3 + (sy + 1) of an entry's mask marks an image
// within the cutoff, d_s = (x_j + s box) - x_i. Cells are periodic in x and y (cell size
// >= rc, coordinates wrapped into the box from its origin) and open in z.
struct PbcGrid {
  double lo[3];      // box origin in x, y; minimum z
  double cell[3];    // cell sizes
  double box[2];
  int64_t dim[3];
};

__device__ __forceinline__ int64_t pcell(double v, double lo, double box, double cell, int64_t dim) {
  double w = v - lo;
  w -= box * floor(w / box);
  int64_t c = (int64_t)floor(w / cell);
  return c < 0 ? 0 : (c >= dim ? dim - 1 : c);
}

__device__ __forceinline__ int64_t zcell(double v, const PbcGrid &g) {
  int64_t c = (int64_t)floor((v - g.lo[2]) / g.cell[2]);
  return c < 0 ? 0 : (c >= g.dim[2] ? g.dim[2] - 1 : c);
}

__device__ __forceinline__ uint32_t image_mask(const double *__restrict__ xyz, int64_t i, int64_t j, double bx,
                                               double by, double rc2) {
  const double xi = xyz[3 * i], yi = xyz[3 * i + 1], zi = xyz[3 * i + 2];
  const double dz = __dsub_rn(xyz[3 * j + 2], zi);
  uint32_t m = 0;
  for (int sx = -1; sx <= 1; ++sx) {
    const double dx = __dsub_rn(__dadd_rn(xyz[3 * j], sx * bx), xi);
    for (int sy = -1; sy <= 1; ++sy) {
      const double dy = __dsub_rn(__dadd_rn(xyz[3 * j + 1], sy * by), yi);
      if (dist2(dx, dy, dz) <= rc2) m |= 1u << ((sx + 1) * 3 + (sy + 1));
    }
  }
  return m;
}

__global__ void k_cell_count_pbc(int64_t n, const double *__restrict__ xyz, PbcGrid g, int32_t *__restrict__ cell_of,
                                 int32_t *__restrict__ count) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int64_t c0 = pcell(xyz[3 * i], g.lo[0], g.box[0], g.cell[0], g.dim[0]);
  const int64_t c1 = pcell(xyz[3 * i + 1], g.lo[1], g.box[1], g.cell[1], g.dim[1]);
  const int64_t c2 = zcell(xyz[3 * i + 2], g);
  const int64_t id = (c0 * g.dim[1] + c1) * g.dim[2] + c2;
  cell_of[i] = (int32_t)id;
  atomicAdd(&count[id], 1);
}

// One thread per atom; every cell is visited once even when a periodic dimension has fewer
// than three cells; an entry is kept when any image is within the cutoff.
__global__ void k_neigh_pbc(int64_t n, const double *__restrict__ xyz, PbcGrid g, double rc2,
                            const int32_t *__restrict__ start, const int32_t *__restrict__ atoms,
                            const int64_t *__restrict__ indptr, int64_t *__restrict__ counts,
                            int32_t *__restrict__ indices) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;   // atoms in cell order
  if (t >= n) return;
  const int64_t i = atoms[t];
  const int64_t c0 = pcell(xyz[3 * i], g.lo[0], g.box[0], g.cell[0], g.dim[0]);
  const int64_t c1 = pcell(xyz[3 * i + 1], g.lo[1], g.box[1], g.cell[1], g.dim[1]);
  const int64_t c2 = zcell(xyz[3 * i + 2], g);
  const int64_t na = g.dim[0] < 3 ? g.dim[0] : 3, nbb = g.dim[1] < 3 ? g.dim[1] : 3;
  int64_t cnt = 0;
  int64_t out = indices ? indptr[i] : 0;
  const int64_t end = indices ? indptr[i + 1] : 0;
  for (int64_t ia = 0; ia < na; ++ia) {
    const int64_t a = g.dim[0] < 3 ? ia : (c0 - 1 + ia + g.dim[0]) % g.dim[0];
    for (int64_t ib = 0; ib < nbb; ++ib) {
      const int64_t b = g.dim[1] < 3 ? ib : (c1 - 1 + ib + g.dim[1]) % g.dim[1];
      for (int64_t c = c2 - 1; c <= c2 + 1; ++c) {
        if (c < 0 || c >= g.dim[2]) continue;
        const int64_t id = (a * g.dim[1] + b) * g.dim[2] + c;
        for (int32_t p = start[id]; p < start[id + 1]; ++p) {
          const int32_t j = atoms[p];
          if (image_mask(xyz, i, j, g.box[0], g.box[1], rc2)) {
            if (indices) {
              if (out < end) indices[out] = j;
              ++out;
            }
            ++cnt;
          }
        }
      }
    }
  }
  if (!indices) counts[i] = cnt;
}

__global__ void k_image_masks(int64_t n, const double *__restrict__ xyz, double bx, double by, double rc2,
                              const int64_t *__restrict__ indptr, const int32_t *__restrict__ indices,
                              uint16_t *__restrict__ images) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  for (int64_t e = indptr[i]; e < indptr[i + 1]; ++e) images[e] = (uint16_t)image_mask(xyz, i, indices[e], bx, by, rc2);
}

// Sorted copy of a row held in LDS (buf[0..len)) into out[0..len), ascending, by one block of 64
// threads (the caller has synchronised after filling buf, which holds kMaxRow + 4 entries). Rows
// of up to 256 entries by rank: every thread counts, for its up to 4 entries, the smaller ones of
// the row, read as 4 per LDS access, and the sorted row is written from LDS in order (one entry
// per access before: 150,000 renumbered rows of 117 in 346 us, now 215). Equal entries leave a place
// unwritten; such a row takes the ranks again with ties by position. Longer rows by a bitonic sort.
__device__ void sort_row_to(int32_t *buf, int32_t *sorted, int len, int32_t *__restrict__ out) {
  const int tid = threadIdx.x, nt = blockDim.x;
  if (len <= 256) {
    const int per = (len + 63) >> 6;
    for (int t = len + tid; t < ((len + 3) & ~3); t += nt) buf[t] = 0x7fffffff;
    int32_t v[4];
    int r[4] = {0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[k] = tid + 64 * k < len ? buf[tid + 64 * k] : 0x7fffffff;
      sorted[tid + 64 * k] = -1;
    }
    __syncthreads();
    auto rank = [&](auto kk) {
      constexpr int K = decltype(kk)::value;
      for (int q = 0; q < len; q += 4) {
        const int4 w = *(const int4 *)(buf + q);
#pragma unroll
        for (int k = 0; k < K; ++k) r[k] += (w.x < v[k]) + (w.y < v[k]) + (w.z < v[k]) + (w.w < v[k]);
      }
    };
    if (per <= 1)
      rank(std::integral_constant<int, 1>());
    else if (per == 2)
      rank(std::integral_constant<int, 2>());
    else
      rank(std::integral_constant<int, 4>());
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (tid + 64 * k < len) sorted[r[k]] = v[k];
    __syncthreads();
    bool hole = false;
    for (int t = tid; t < len; t += nt) hole |= sorted[t] < 0;
    if (__ballot(hole)) {   // one wave: uniform
      __syncthreads();
      for (int t = tid; t < len; t += nt) {
        const int32_t x = buf[t];
        int at = 0;
        for (int q = 0; q < len; ++q) at += (buf[q] < x) | ((buf[q] == x) & (q < t));
        sorted[at] = x;
      }
      __syncthreads();
    }
    for (int t = tid; t < len; t += nt) out[t] = sorted[t];
    return;
  }
  int p2 = 1;
  while (p2 < len) p2 <<= 1;
  for (int t = len + tid; t < p2; t += nt) buf[t] = 0x7fffffff;
  __syncthreads();
  for (int k = 2; k <= p2; k <<= 1) {
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int t = tid; t < p2; t += nt) {
        const int ixj = t ^ j;
        if (ixj > t) {
          const bool up = (t & k) == 0;
          const int32_t x = buf[t], y = buf[ixj];
          if ((x > y) == up) {
            buf[t] = y;
            buf[ixj] = x;
          }
        }
      }
      __syncthreads();
    }
  }
  for (int t = tid; t < len; t += nt) out[t] = buf[t];
}

// One 64-thread block per row: the row's columns sorted ascending in place.
__global__ void __launch_bounds__(64) k_sort_rows(int64_t n, const int64_t *__restrict__ indptr,
                                                   int32_t *__restrict__ indices, int32_t *__restrict__ overflow) {
  __shared__ __align__(16) int32_t buf[kMaxRow + 4];
  __shared__ int32_t sorted[256];
  const int64_t row = blockIdx.x;
  if (row >= n) return;
  const int64_t b = indptr[row], e = indptr[row + 1];
  const int len = (int)(e - b);
  if (len > kMaxRow) {
    if (threadIdx.x == 0) atomicMax(overflow, len);
    return;
  }
  for (int t = threadIdx.x; t < len; t += blockDim.x) buf[t] = indices[b + t];
  __syncthreads();
  sort_row_to(buf, sorted, len, indices + b);
}

// counts[i] = length of row order[i] of the source CSR
__global__ void k_perm_counts(int64_t n, const int64_t *__restrict__ indptr, const int32_t *__restrict__ order,
                              int64_t *__restrict__ counts) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int64_t o = order[i];
  counts[i] = indptr[o + 1] - indptr[o];
}

// One block per new row: the columns of source row order[row], renumbered by undo (old index
// -> new index), sorted ascending (sort_row_to).
__global__ void __launch_bounds__(64) k_permute_sort_rows(int64_t n, const int64_t *__restrict__ indptr,
                                                           const int32_t *__restrict__ indices,
                                                           const int32_t *__restrict__ order,
                                                           const int64_t *__restrict__ undo,
                                                           const int64_t *__restrict__ out_ptr,
                                                           int32_t *__restrict__ out_idx,
                                                           int32_t *__restrict__ overflow) {
  __shared__ __align__(16) int32_t buf[kMaxRow + 4];
  __shared__ int32_t sorted[256];
  const int64_t row = blockIdx.x;
  if (row >= n) return;
  const int64_t o = order[row];
  const int64_t b = indptr[o];
  const int len = (int)(indptr[o + 1] - b);
  if (len > kMaxRow) {
    if (threadIdx.x == 0) atomicMax(overflow, len);
    return;
  }
  for (int t = threadIdx.x; t < len; t += blockDim.x) buf[t] = (int32_t)undo[indices[b + t]];
  __syncthreads();
  sort_row_to(buf, sorted, len, out_idx + out_ptr[row]);
}

// One 64-lane wave per row: H_ij = -d d^T / r^2 for j != i (r^2 > 0); the diagonal
// block is minus the sum of the row's off-diagonal blocks plus plus_i * I.
__global__ void __launch_bounds__(256) k_assemble(int64_t n, const double *__restrict__ xyz, double plus_i,
                                                   const int64_t *__restrict__ rowptr, const int32_t *__restrict__ col,
                                                   const uint16_t *__restrict__ images, double bx, double by,
                                                   double *__restrict__ v64, float *__restrict__ v32,
                                                   double *__restrict__ diag) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 6;
  if (row >= n) return;
  const double xi = xyz[3 * row], yi = xyz[3 * row + 1], zi = xyz[3 * row + 2];
  double s[6] = {0, 0, 0, 0, 0, 0};  // xx xy xz yy yz zz of sum d d^T / r^2
  int64_t selfpos = -1;
  const int64_t b0 = rowptr[row], b1 = rowptr[row + 1];
  for (int64_t b = b0 + lane; b < b1; b += 64) {
    int32_t j = col[b];
    double h[9];
    if (j == row) {
      selfpos = b;
      continue;
    }
    if (!images) {
      double dx = __dsub_rn(xyz[3 * (int64_t)j], xi), dy = __dsub_rn(xyz[3 * (int64_t)j + 1], yi),
             dz = __dsub_rn(xyz[3 * (int64_t)j + 2], zi);
      double r2 = dist2(dx, dy, dz);
      double c = r2 > 0.0 ? -1.0 / r2 : 0.0;
      double d[3] = {dx, dy, dz};
      for (int p = 0; p < 3; ++p)
        for (int q = 0; q < 3; ++q) h[3 * p + q] = d[p] * d[q] * c;
    } else {
      // sum over the images of j within the cutoff
      for (int t = 0; t < 9; ++t) h[t] = 0.0;
      const uint32_t m = images[b];
      const double dz = __dsub_rn(xyz[3 * (int64_t)j + 2], zi);
      for (int bit = 0; bit < 9; ++bit) {
        if (!((m >> bit) & 1u)) continue;
        const double sx = (double)(bit / 3 - 1), sy = (double)(bit % 3 - 1);
        const double dx = __dsub_rn(__dadd_rn(xyz[3 * (int64_t)j], sx * bx), xi);
        const double dy = __dsub_rn(__dadd_rn(xyz[3 * (int64_t)j + 1], sy * by), yi);
        const double r2 = dist2(dx, dy, dz);
        const double c = r2 > 0.0 ? -1.0 / r2 : 0.0;
        const double d[3] = {dx, dy, dz};
        for (int p = 0; p < 3; ++p)
          for (int q = 0; q < 3; ++q) h[3 * p + q] += d[p] * d[q] * c;
      }
    }
    s[0] -= h[0];
    s[1] -= h[1];
    s[2] -= h[2];
    s[3] -= h[4];
    s[4] -= h[5];
    s[5] -= h[8];
    if (v64)
      for (int t = 0; t < 9; ++t) v64[9 * b + t] = h[t];
    if (v32)
      for (int t = 0; t < 9; ++t) v32[9 * b + t] = (float)h[t];
  }
  // deterministic butterfly reduction over the wave
  for (int off = 32; off > 0; off >>= 1)
    for (int t = 0; t < 6; ++t) s[t] += __shfl_xor(s[t], off, 64);
  // the lane holding the self block writes it
  if (selfpos >= 0) {
    double h[9] = {s[0] + plus_i, s[1], s[2], s[1], s[3] + plus_i, s[4], s[2], s[4], s[5] + plus_i};
    if (v64)
      for (int t = 0; t < 9; ++t) v64[9 * selfpos + t] = h[t];
    if (v32)
      for (int t = 0; t < 9; ++t) v32[9 * selfpos + t] = (float)h[t];
  }
  if (diag && lane == 0) {
    diag[3 * row] = s[0] + plus_i;
    diag[3 * row + 1] = s[3] + plus_i;
    diag[3 * row + 2] = s[5] + plus_i;
  }
}

// ---- cluster layout of the matrix-free operator --------------------------------------
// Atoms are grouped into clusters of kClusterAtoms that are compact in space: cells of
// cell_xy x cell_xy x cell_z, numbered column-major (x, y column, then z inside the column),
// atoms in a cell by index, cut into groups of 4; the groups are numbered by their smallest
// neighbour index, so consecutive clusters gather from one band of the vectors. Each cluster
// lists the union of its atoms' neighbour rows once, as (j, mask) with mask bit t set when j
// is a neighbour of the cluster's atom t (j itself excluded), so the product gathers a
// neighbour's coordinates and vector entries once per cluster instead of once per atom.
constexpr int kClusterAtoms = 4;
constexpr int kMaxUnion = 4096;  // row entries one cluster may gather (LDS sort capacity)

struct CGrid {
  double lo[3];
  double inv[3];  // 1 / cell size per axis
  int64_t dim[3];
};

__global__ void k_cl_cell(int64_t n, const double *__restrict__ xyz, CGrid g, int32_t *__restrict__ cell_of,
                          int32_t *__restrict__ count) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  int64_t c[3];
  for (int a = 0; a < 3; ++a) c[a] = cell_coord(xyz[3 * i + a], g.lo[a], g.inv[a], g.dim[a]);
  const int64_t id = (c[0] * g.dim[1] + c[1]) * g.dim[2] + c[2];
  cell_of[i] = (int32_t)id;
  atomicAdd(&count[id], 1);
}

// One thread per cell: insertion sort of the cell's atoms by index (cells hold a few atoms),
// which makes the order independent of the atomic fill order.
__global__ void k_cell_isort(int64_t ncell, const int32_t *__restrict__ start, int32_t *__restrict__ atoms) {
  const int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (c >= ncell) return;
  const int32_t b = start[c], e = start[c + 1];
  for (int32_t p = b + 1; p < e; ++p) {
    const int32_t v = atoms[p];
    int32_t q = p - 1;
    while (q >= b && atoms[q] > v) {
      atoms[q + 1] = atoms[q];
      --q;
    }
    atoms[q + 1] = v;
  }
}

__global__ void k_cl_atoms(int64_t n, int64_t slots, const int32_t *__restrict__ atoms,
                           int32_t *__restrict__ cluster_atoms) {
  const int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (q < slots) cluster_atoms[q] = q < n ? atoms[q] : -1;
}

// Squared distance of atoms i and j as the cluster product computes it (d = p_j - p_i, the
// same FMAs): a pair at r2 = 0 (coincident atoms, whose term the reference masks) gets no
// list bit, so the product needs no test of its own.
__device__ __forceinline__ double cl_pair_r2(const double *__restrict__ xyz, int64_t i, int64_t j) {
  const double d0 = xyz[3 * j] - xyz[3 * i], d1 = xyz[3 * j + 1] - xyz[3 * i + 1], d2 = xyz[3 * j + 2] - xyz[3 * i + 2];
  return __builtin_fma(d2, d2, __builtin_fma(d1, d1, d0 * d0));
}

// One block per cluster. The rows of its atoms (each in ascending column order, as the
// neighbour search and the renumbering write them) are merged into keys (j << 3 | t) in
// ascending order in LDS, and each run of equal j becomes one entry with the OR of its atom
// bits.
// Count pass (FILL = false): counts[c] = entries, base[c] = smallest j; overflow bit 1 =
// more than kMaxUnion row entries, bit 2 = the union spans 2^24 columns or more. With
// prov_ptr given it also writes the entries, at prov_ptr[c] (room for all of the cluster's row
// entries), for a later copy into the final layout.
// Fill pass: entries[cl_ptr[c] + r] = ((j - base[c]) << 8) | mask, ascending j.
template <bool FILL>
__global__ void __launch_bounds__(256) k_cl_union(int64_t n, int64_t ncl, const double *__restrict__ xyz,
                                                   const int64_t *__restrict__ rowptr,
                                                   const int32_t *__restrict__ col,
                                                   const int32_t *__restrict__ cluster_atoms,
                                                   const int64_t *__restrict__ cl_ptr, int32_t *__restrict__ base,
                                                   int64_t *__restrict__ counts, uint32_t *__restrict__ entries,
                                                   int32_t *__restrict__ overflow,
                                                   const int64_t *__restrict__ prov_ptr = nullptr) {
  __shared__ uint64_t key[kMaxUnion];
  __shared__ int32_t val[kMaxUnion];
  __shared__ int32_t part[256];
  __shared__ int64_t rb[kClusterAtoms], rl[kClusterAtoms + 1];
  __shared__ int32_t ca[kClusterAtoms];
  __shared__ int32_t s_min, s_max, s_bad;
  const int64_t c = blockIdx.x;
  const int tid = threadIdx.x;
  if (tid == 0) {
    int64_t acc = 0;
    for (int t = 0; t < kClusterAtoms; ++t) {
      const int32_t a = cluster_atoms[kClusterAtoms * c + t];
      ca[t] = a;
      const int64_t b = a >= 0 ? rowptr[a] : 0, e = a >= 0 ? rowptr[a + 1] : 0;
      rb[t] = b;
      rl[t] = acc;
      acc += e - b;
    }
    rl[kClusterAtoms] = acc;
    s_min = 0;
    s_max = 0;
    s_bad = 0;
  }
  __syncthreads();
  const int64_t total64 = rl[kClusterAtoms];
  if (total64 > kMaxUnion) {  // uniform over the block
    if (tid == 0) {
      atomicOr(overflow, 1);
      if (!FILL) counts[c] = 0;
    }
    return;
  }
  const int total = (int)total64;
  // the four rows (ascending columns) into val[]; each entry's place in the merged order is
  // its index in its own row plus, for every other row, the entries below it (equal columns
  // of earlier rows count as below), found by binary search: the keys (j << 3 | t) come out
  // in ascending order, as a sort of them would give. A row out of order sets overflow bit 4.
  for (int e = tid; e < total; e += blockDim.x) {
    int t = 0;
    while (e >= rl[t + 1]) ++t;
    val[e] = col[rb[t] + (e - rl[t])];
  }
  __syncthreads();
  // rows out of order would make the ranks collide and leave keys unwritten, and a column
  // outside [0, n) would address coordinates out of bounds: the block stops here, before any
  // rank is formed (uniform exit)
  for (int e = tid; e < total; e += blockDim.x) {
    int t = 0;
    while (e >= rl[t + 1]) ++t;
    if ((e > rl[t] && val[e - 1] >= val[e]) || val[e] < 0 || val[e] >= n) s_bad = 1;
  }
  __syncthreads();
  if (s_bad) {
    if (tid == 0) {
      atomicOr(overflow, 4);
      if (!FILL) counts[c] = 0;
    }
    return;
  }
  for (int e = tid; e < total; e += blockDim.x) {
    int t = 0;
    while (e >= rl[t + 1]) ++t;
    const int32_t j = val[e];
    int rank = e - (int)rl[t];
    for (int u = 0; u < kClusterAtoms; ++u) {
      if (u == t) continue;
      int lo = (int)rl[u], hi = (int)rl[u + 1];
      while (lo < hi) {
        const int m = (lo + hi) >> 1;
        const int32_t x = val[m];
        if (u < t ? x <= j : x < j)
          lo = m + 1;
        else
          hi = m;
      }
      rank += lo - (int)rl[u];
    }
    key[rank] = ((uint64_t)(uint32_t)j << 3) | (uint64_t)t;
  }
  __syncthreads();
  // runs of equal j: the run's first element carries the mask (0 = nothing to emit)
  const int chunk = (total + 255) / 256;
  const int e0 = tid * chunk, e1 = min(total, e0 + chunk);
  int cnt = 0;
  for (int e = e0; e < e1; ++e) {
    const uint32_t j = (uint32_t)(key[e] >> 3);
    int32_t m = 0;
    if (e == 0 || (uint32_t)(key[e - 1] >> 3) != j) {
      for (int f = e; f < total && (uint32_t)(key[f] >> 3) == j; ++f) {
        const int t = (int)(key[f] & 7);
        if ((uint32_t)ca[t] != j && cl_pair_r2(xyz, ca[t], j) > 0.0) m |= 1 << t;
      }
    }
    val[e] = m;
    cnt += m != 0;
  }
  part[tid] = cnt;
  __syncthreads();
  for (int off = 1; off < 256; off <<= 1) {
    const int v = tid >= off ? part[tid - off] : 0;
    __syncthreads();
    part[tid] += v;
    __syncthreads();
  }
  const int before = part[tid] - cnt, emitted = part[255];
  if (!FILL) {
    if (cnt > 0) {
      int first = -1, last = -1;
      for (int e = e0; e < e1; ++e)
        if (val[e]) {
          if (first < 0) first = e;
          last = e;
        }
      if (before == 0) s_min = (int32_t)(key[first] >> 3);
      if (before + cnt == emitted) s_max = (int32_t)(key[last] >> 3);
    }
    __syncthreads();
    if (tid == 0) {
      counts[c] = emitted;
      base[c] = s_min;
      if (emitted > 0 && (int64_t)s_max - (int64_t)s_min >= ((int64_t)1 << 24)) atomicOr(overflow, 2);
    }
    if (prov_ptr) {
      const int64_t out = prov_ptr[c] + before;
      const uint32_t b0 = (uint32_t)s_min;
      int r = 0;
      for (int e = e0; e < e1; ++e)
        if (val[e]) entries[out + r++] = (((uint32_t)(key[e] >> 3) - b0) << 8) | (uint32_t)val[e];
    }
    return;
  }
  const int64_t out = cl_ptr[c] + before;
  const uint32_t b0 = (uint32_t)base[c];
  int r = 0;
  for (int e = e0; e < e1; ++e)
    if (val[e]) entries[out + r++] = (((uint32_t)(key[e] >> 3) - b0) << 8) | (uint32_t)val[e];
}

// Sort keys of the clusters: smallest neighbour in the high word, cluster index in the low.
__global__ void k_cl_keys(int64_t ncl, const int32_t *__restrict__ base, uint64_t *__restrict__ key) {
  const int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (c < ncl) key[c] = ((uint64_t)(uint32_t)base[c] << 32) | (uint64_t)c;
}

// Clusters renumbered: slot c' takes cluster perm[c'] = low word of the c'-th sorted key
// (atoms, list length, base).
__global__ void k_cl_permute(int64_t ncl, const uint64_t *__restrict__ perm, const int32_t *__restrict__ atoms_in,
                             const int64_t *__restrict__ counts_in, const int32_t *__restrict__ base_in,
                             int32_t *__restrict__ atoms_out, int64_t *__restrict__ counts_out,
                             int32_t *__restrict__ base_out) {
  const int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (c >= ncl) return;
  const int64_t src = (int64_t)(perm[c] & 0xffffffffu);
  for (int t = 0; t < kClusterAtoms; ++t) atoms_out[kClusterAtoms * c + t] = atoms_in[kClusterAtoms * src + t];
  counts_out[c] = counts_in[src];
  base_out[c] = base_in[src];
}

// tot[c] = entries of the rows of cluster c's atoms (room for its list before the union)
__global__ void k_cl_totals(int64_t ncl, const int32_t *__restrict__ cluster_atoms,
                            const int64_t *__restrict__ rowptr, int64_t *__restrict__ tot) {
  const int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (c >= ncl) return;
  int64_t s = 0;
  for (int t = 0; t < kClusterAtoms; ++t) {
    const int32_t a = cluster_atoms[kClusterAtoms * c + t];
    if (a >= 0) s += rowptr[a + 1] - rowptr[a];
  }
  tot[c] = s;
}

// Final layout from the count pass's provisional lists: cluster c' (new numbering) takes the
// list of cluster perm[c'] (old numbering), written at prov_ptr of the old cluster.
__global__ void __launch_bounds__(256) k_cl_copy(int64_t ncl, const uint64_t *__restrict__ perm,
                                                 const int64_t *__restrict__ prov_ptr,
                                                 const uint32_t *__restrict__ prov,
                                                 const int64_t *__restrict__ cl_ptr, uint32_t *__restrict__ entries) {
  const int64_t c = blockIdx.x;
  const int64_t src = prov_ptr[(int64_t)(perm[c] & 0xffffffffu)];
  const int64_t dst = cl_ptr[c], len = cl_ptr[c + 1] - dst;
  for (int64_t e = threadIdx.x; e < len; e += blockDim.x) entries[dst + e] = prov[src + e];
}

// ---- record form of the cluster layout (the operator's Chebyshev recurrence) ----
// rec[6 q .. 6 q + 2] = coordinates of slot q = 4 c + t (atom cluster_atoms[q]; zeros for a
// padding slot), rec[6 q + 3 .. 6 q + 5] = 0 (the vector part, written by the pack and the
// product); slot_of[atom] = its slot.
__global__ void k_rec_coords(int64_t slots, const int32_t *__restrict__ cluster_atoms, const double *__restrict__ xyz,
                             double *__restrict__ rec, int32_t *__restrict__ slot_of) {
  const int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (q >= slots) return;
  const int32_t at = cluster_atoms[q];
  for (int k = 0; k < 3; ++k) {
    rec[6 * q + k] = at >= 0 ? xyz[3 * (int64_t)at + k] : 0.0;
    rec[6 * q + 3 + k] = 0.0;
  }
  if (at >= 0) slot_of[at] = (int32_t)q;
}

// One block per cluster: its list rewritten as 48 (slot of j) | mask -- the byte offset of
// j's 48-byte record, whose low 4 bits are zero, carrying the mask -- and sorted ascending
// (bitonic sort in LDS; a list holds fewer than kMaxUnion entries).
__global__ void __launch_bounds__(256) k_rec_lists(int64_t ncl, const int64_t *__restrict__ cl_ptr,
                                                    const int32_t *__restrict__ base,
                                                    const uint32_t *__restrict__ entries,
                                                    const int32_t *__restrict__ slot_of, uint32_t *__restrict__ out) {
  __shared__ uint32_t key[kMaxUnion];
  const int64_t c = blockIdx.x;
  const int64_t e0 = cl_ptr[c];
  const int len = (int)(cl_ptr[c + 1] - e0);
  const uint32_t b0 = (uint32_t)base[c];
  int p2 = 1;
  while (p2 < len) p2 <<= 1;
  for (int e = threadIdx.x; e < p2; e += blockDim.x) {
    uint32_t k = 0xffffffffu;
    if (e < len) {
      const uint32_t w = entries[e0 + e];
      k = 48u * (uint32_t)slot_of[b0 + (w >> 8)] | (w & 15u);
    }
    key[e] = k;
  }
  __syncthreads();
  for (int k = 2; k <= p2; k <<= 1) {
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int t = threadIdx.x; t < p2; t += blockDim.x) {
        const int ixj = t ^ j;
        if (ixj > t) {
          const bool up = (t & k) == 0;
          const uint32_t a = key[t], b = key[ixj];
          if ((a > b) == up) {
            key[t] = b;
            key[ixj] = a;
          }
        }
      }
      __syncthreads();
    }
  }
  for (int e = threadIdx.x; e < len; e += blockDim.x) out[e0 + e] = key[e];
}

// ---- tile form of the matrix-free operator (the operator's Chebyshev recurrence) ----
// Atoms are numbered by slots: sorted along columns of side x side in x and y (boustrophedon
// over the columns and along z, so that consecutive tiles stay close across a turn), every
// column cut into equal tiles of at most TA atoms, inside a tile by falling row length (a wave
// of the product runs as many passes as its longest row needs). A tile that spans two columns
// would be long and its union large (up to 1.6 times, and beyond the limit where a column
// crosses several parts of an assembly); the equal shares leave 3% of the slots empty in a
// 300,000-atom globule. A tile lists the union of its atoms' neighbours once; each atom then
// lists its own as 16-bit offsets into that union.

// Order of the atoms: (column, place along it) in 64 bits, sorted stably with the atom index.
__global__ void k_tile_keys(int64_t n, const double *__restrict__ xyz, CGrid g, double zscale,
                            uint64_t *__restrict__ key, int32_t *__restrict__ atom) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int64_t cx = cell_coord(xyz[3 * i], g.lo[0], g.inv[0], g.dim[0]);
  int64_t cy = cell_coord(xyz[3 * i + 1], g.lo[1], g.inv[1], g.dim[1]);
  if (cx & 1) cy = g.dim[1] - 1 - cy;
  const int64_t c = cx * g.dim[1] + cy;
  const double f = (xyz[3 * i + 2] - g.lo[2]) * zscale;   // 0 .. 2^32 - 1
  uint32_t z = f < 4294967295.0 ? (uint32_t)f : 0xffffffffu;
  if (c & 1) z = ~z;
  key[i] = ((uint64_t)c << 32) | z;
  atom[i] = (int32_t)i;
}

// head[i] = 1 where a new column begins in the sorted keys
__global__ void k_tile_heads(int64_t n, const uint64_t *__restrict__ key, int32_t *__restrict__ head) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) head[i] = i == 0 || (key[i] >> 32) != (key[i - 1] >> 32);
}

// first[c] = where column c begins (first[columns] = n); cidx: exclusive scan of head
__global__ void k_tile_first(int64_t n, const int32_t *__restrict__ head, const int32_t *__restrict__ cidx,
                             int32_t *__restrict__ first) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n && head[i]) first[cidx[i]] = (int32_t)i;
  if (i == 0) first[cidx[n]] = (int32_t)n;
}

// tiles of column c (0 beyond the last column)
__global__ void k_tile_column(int64_t n, int TA, const int32_t *__restrict__ cidx, const int32_t *__restrict__ first,
                              int32_t *__restrict__ tiles) {
  const int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (c < n) tiles[c] = c < cidx[n] ? (first[c + 1] - first[c] + TA - 1) / TA : 0;
}

// tile_start of every tile of column c: the column's atoms in equal shares
__global__ void k_tile_cut(int64_t n, const int32_t *__restrict__ cidx, const int32_t *__restrict__ first,
                           const int32_t *__restrict__ base, int32_t *__restrict__ tile_start) {
  const int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (c >= cidx[n]) return;
  const int64_t b = first[c], len = first[c + 1] - b, t0 = base[c], K = base[c + 1] - t0;
  for (int64_t k = 0; k < K; ++k) tile_start[t0 + k] = (int32_t)(b + len * k / K);
  if (c == cidx[n] - 1) tile_start[t0 + K] = (int32_t)n;
}

// The image masks of an entry with a term: bits of the images at a nonzero distance (open
// boundaries: bit 4, the unshifted one). far |= 1 when a distance leaves the range in which
// the product's float32 reciprocal seed is normal.
template <bool PBC>
__device__ __forceinline__ uint32_t tile_images(const double *__restrict__ xyz, int64_t i, int64_t j,
                                                const uint16_t *__restrict__ images, int64_t e, double bx, double by,
                                                int &far) {
  uint32_t m = PBC ? (uint32_t)images[e] & 511u : 16u, keep = 0;
  while (m) {
    const int bit = __ffs(m) - 1;
    m &= m - 1;
    const double sx = PBC ? (double)(bit / 3 - 1) * bx : 0.0, sy = PBC ? (double)(bit % 3 - 1) * by : 0.0;
    const double d0 = (xyz[3 * j] + sx) - xyz[3 * i], d1 = (xyz[3 * j + 1] + sy) - xyz[3 * i + 1];
    const double d2 = xyz[3 * j + 2] - xyz[3 * i + 2];
    const double r2 = __builtin_fma(d2, d2, __builtin_fma(d1, d1, d0 * d0));
    if (r2 > 0.0) {
      keep |= 1u << bit;
      if (!(r2 > 1e-30 && r2 < 1e30)) far = 1;
    }
  }
  return keep;
}

// cnt[i] = terms of atom i (entries times their images); one 16-lane group per row. Flags: bit 0 more than `most`
// terms (so many different ones are more than a union holds; repeated columns would exceed k_tile_fill's places),
// bit 3 a column outside [0, n), bit 4 a distance outside the float32 seed's range.
template <bool PBC>
__global__ void __launch_bounds__(256) k_tile_count(int64_t n, const double *__restrict__ xyz,
                                                    const int64_t *__restrict__ rowptr,
                                                    const int32_t *__restrict__ col,
                                                    const uint16_t *__restrict__ images, double bx, double by,
                                                    int most, int32_t *__restrict__ cnt,
                                                    int32_t *__restrict__ flags) {
  const int64_t i = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 4;
  const int lane = threadIdx.x & 15;
  if (i >= n) return;
  int32_t c = 0;
  int far = 0;
  for (int64_t e = rowptr[i] + lane; e < rowptr[i + 1]; e += 16) {
    const int32_t j = col[e];
    if (j < 0 || j >= n) {
      atomicOr(flags, 8);
      continue;
    }
    c += __popc(tile_images<PBC>(xyz, i, j, images, e, bx, by, far));
  }
  if (far) atomicOr(flags, 16);
#pragma unroll
  for (int off = 8; off > 0; off >>= 1) c += __shfl_xor(c, off, 16);
  if (lane == 0) {
    cnt[i] = c;
    if (c > most) atomicOr(flags, 1);
  }
}

// One 64-thread block per tile: its atoms by falling term count (ties by place), the slot of
// every atom, and per wave of 64 / G atoms its passes (terms of its longest row / G) and its
// blocks of 8 passes.
__global__ void __launch_bounds__(64) k_tile_slots(int TA, int G, const int32_t *__restrict__ sorted,
                                                   const int32_t *__restrict__ tile_start,
                                                   const int32_t *__restrict__ cnt, int32_t *__restrict__ tile_atoms,
                                                   int32_t *__restrict__ slot_of, int32_t *__restrict__ passes,
                                                   int32_t *__restrict__ blocks) {
  __shared__ int32_t ca[64], cc[64];
  const int64_t t = blockIdx.x;
  const int q = threadIdx.x;
  const int64_t at = (int64_t)tile_start[t] + q;
  int32_t a = -1, c = -1;
  if (q < TA && at < tile_start[t + 1]) {
    a = sorted[at];
    c = cnt[a];
  }
  ca[q] = c;
  __syncthreads();
  int r = 0;
  if (q < TA) {
    for (int p = 0; p < TA; ++p) r += ca[p] > c || (ca[p] == c && p < q);
    tile_atoms[t * TA + r] = a;
    if (a >= 0) slot_of[a] = (int32_t)(t * TA + r);
    cc[r] = c;
  }
  __syncthreads();
  const int AW = 64 / G, NW = TA / AW;
  if (q < NW) {
    const int32_t top = cc[q * AW];           // falling: the wave's first atom has the most terms
    const int32_t p = top > 0 ? (top + G - 1) / G : 0;
    passes[t * NW + q] = p;
    blocks[t * NW + q] = (p + 7) / 8;
  }
}

// waves[w] = (first block, passes) of wave w
__global__ void k_tile_waves(int64_t nw, const int32_t *__restrict__ ptr, const int32_t *__restrict__ passes,
                             int2 *__restrict__ waves) {
  const int64_t w = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (w < nw) waves[w] = make_int2(ptr[w], passes[w]);
}

// Place (pass, lane of the atom's G) of the rho-th term whose union place has residue r mod 16, for
// the atom at place a of its tile. The product's 16-byte LDS reads serve a half wave in two groups
// of 16 lanes, lanes {0-3, 12-15, 20-23, 24-27} and the others (measured: these are the only sets
// of 16 that conflict among themselves), and a record's three reads meet banks by its place mod 16
// (48 bytes are three groups of four of the 64 banks). So the 16 lanes of a group take 16
// different residues in every pass: with G = 8 a group holds 4 lanes of 4 atoms, which take the
// residues by quarters, another quarter each pass; with G = 16 8 lanes of 2 atoms, by halves;
// with G = 32 the 16 lanes of one atom. Terms beyond a residue's places fill the gaps of others.
__device__ __forceinline__ int2 tile_place(int G, int r, int rho, int a) {
  const int half = rho & 1, c = rho >> 1;
  if (G == 8) return make_int2(4 * c + (((r >> 2) - a) & 3), (r & 3) + 4 * half);
  if (G == 16) {
    const int q = r & 7;
    return make_int2(2 * c + (((r >> 3) ^ a) & 1), half ? 4 + q : (q < 4 ? q : q + 8));
  }
  // lanes of the two groups in order: r-th lane of group `half`
  const int g4 = r >> 2;
  const int base = half ? (g4 == 0 ? 4 : g4 == 1 ? 8 : g4 == 2 ? 16 : 28) : (g4 == 0 ? 0 : g4 == 1 ? 12 : g4 == 2 ? 20 : 24);
  return make_int2(c, base + (r & 3));
}

constexpr int kTileHash = 4096;   // slots of the union's hash table: at least 3 x the largest union

// One block per tile. The (neighbour slot, image) words of its rows go into an LDS hash
// table; the distinct ones, sorted, are the tile's union (written as 48 slot | image: the
// byte offset of the neighbour's record, the image in its low 4 bits). Then a wave per row
// writes its terms as 16-bit byte offsets 48 p of their places p in the union, each to its pass
// and lane (tile_place), 8 passes to a block of 64 lanes x 16 bytes. Places that a row does not
// fill name the atom's own dummy record 48 (union + atom), whose term is zero. flags bit 0: the
// union exceeds ucap.
template <bool PBC>
__global__ void __launch_bounds__(256) k_tile_fill(int64_t n, int TA, int G, const double *__restrict__ xyz,
                                                   const int64_t *__restrict__ rowptr,
                                                   const int32_t *__restrict__ col,
                                                   const uint16_t *__restrict__ images, double bx, double by,
                                                   const int32_t *__restrict__ tile_atoms,
                                                   const int32_t *__restrict__ slot_of, const int2 *__restrict__ waves,
                                                   int ucap, int32_t *__restrict__ ulen, uint32_t *__restrict__ ulist,
                                                   uint16_t *__restrict__ pairs, int32_t *__restrict__ flags,
                                                   int32_t *__restrict__ umax) {
  __shared__ uint32_t hkey[kTileHash];
  __shared__ uint16_t hpos[kTileHash];
  __shared__ uint32_t list[2048];
  __shared__ uint32_t taken[4][64];      // a wave's places in use: at most 1,349 terms (k_tile_count) + G < 2,048
  __shared__ uint16_t spills[4][1408];   // at most its terms
  __shared__ int s_n;
  const int64_t t = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  constexpr uint32_t kEmpty = 0xffffffffu;
  for (int q = tid; q < kTileHash; q += 256) hkey[q] = kEmpty;
  if (tid == 0) s_n = 0;
  __syncthreads();
  auto place = [](uint32_t k) { return (k * 2654435761u) >> 20; };   // 12 bits
  int far = 0;
  for (int a = w; a < TA; a += 4) {
    const int32_t i = tile_atoms[t * TA + a];
    if (i < 0) continue;
    for (int64_t e = rowptr[i] + lane; e < rowptr[i + 1]; e += 64) {
      const int32_t j = col[e];
      uint32_t m = tile_images<PBC>(xyz, i, j, images, e, bx, by, far);
      while (m) {
        const int bit = __ffs(m) - 1;
        m &= m - 1;
        const uint32_t k = ((uint32_t)slot_of[j] << 4) | (uint32_t)bit;
        uint32_t h = place(k);
        // the table never fills: a thread stops once more than ucap words are in, so at most
        // ucap + 256 < kTileHash are
        while (*(volatile int *)&s_n <= ucap) {
          const uint32_t old = atomicCAS(&hkey[h], kEmpty, k);
          if (old == k) break;
          if (old == kEmpty) {
            atomicAdd(&s_n, 1);
            break;
          }
          h = (h + 1) & (kTileHash - 1);
        }
      }
    }
  }
  __syncthreads();
  const int ul = s_n;
  if (ul > ucap) {   // uniform
    if (tid == 0) {
      atomicOr(flags, 1);
      ulen[t] = 0;
    }
    return;
  }
  __syncthreads();
  if (tid == 0) s_n = 0;
  __syncthreads();
  for (int q = tid; q < kTileHash; q += 256)
    if (hkey[q] != kEmpty) list[atomicAdd(&s_n, 1)] = hkey[q];
  int p2 = 1;
  while (p2 < ul) p2 <<= 1;
  __syncthreads();
  for (int q = ul + tid; q < p2; q += 256) list[q] = kEmpty;
  __syncthreads();
  for (int k = 2; k <= p2; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int q = tid; q < p2 / 2; q += 256) {
        const int lo = 2 * j * (q / j) + q % j, hi = lo + j;
        const uint32_t x = list[lo], y = list[hi];
        if ((x > y) == ((lo & k) == 0)) {
          list[lo] = y;
          list[hi] = x;
        }
      }
      __syncthreads();
    }
  for (int q = tid; q < ul; q += 256) {
    const uint32_t k = list[q];
    uint32_t h = place(k);
    while (hkey[h] != k) h = (h + 1) & (kTileHash - 1);
    hpos[h] = (uint16_t)q;
    ulist[t * ucap + q] = 48u * (k >> 4) | (k & 15u);
  }
  if (tid == 0) {
    ulen[t] = ul;
    atomicMax(umax, ul);
  }
  __syncthreads();
  const int AW = 64 / G, NW = TA / AW;
  const uint64_t below = ((uint64_t)1 << lane) - 1;
  for (int a = w; a < TA; a += 4) {
    const int32_t i = tile_atoms[t * TA + a];
    const int2 wv = waves[t * NW + a / AW];
    const int passes = wv.y, slots = passes * G;
    uint16_t *out = pairs + 512 * (int64_t)wv.x;
    const int l0 = (a % AW) * G;
    auto put = [&](int pass, int l, uint32_t p) {
      out[((pass >> 3) * 64 + l0 + l) * 8 + (pass & 7)] = (uint16_t)(48u * p);
    };
    taken[w][lane] = 0;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    int seen = 0, spilled = 0;   // lane r < 16: terms of residue r so far; terms without a place of their own
    if (i >= 0) {
      const int64_t e1 = rowptr[i + 1];
      for (int64_t e0 = rowptr[i]; e0 < e1; e0 += 64) {
        const int64_t e = e0 + lane;
        uint32_t m = 0;
        uint32_t s = 0;
        if (e < e1) {
          const int32_t j = col[e];
          m = tile_images<PBC>(xyz, i, j, images, e, bx, by, far);
          s = (uint32_t)slot_of[j];
        }
        while (true) {   // one image per lane at a time
          const uint64_t has = __ballot(m != 0);
          if (!has) break;
          uint32_t p = 0;
          if (m) {
            const uint32_t k = (s << 4) | (uint32_t)(__ffs(m) - 1);
            uint32_t h = place(k);
            while (hkey[h] != k) h = (h + 1) & (kTileHash - 1);
            p = hpos[h];
          }
          const uint32_t r = p & 15u;
          uint64_t same = has, mine = has;   // lanes of this lane's residue; of residue `lane`
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const uint64_t bal = __ballot((r >> q) & 1u);
            same &= (r >> q) & 1u ? bal : ~bal;
            mine &= (lane >> q) & 1 ? bal : ~bal;
          }
          const int rho = __shfl(seen, (int)r, 64) + __popcll(same & below);
          seen += __popcll(mine);
          const int2 at = tile_place(G, (int)r, rho, a);
          const bool spill = m && at.x >= passes;
          if (m && !spill) {
            put(at.x, at.y, p);
            const int q = at.x * G + at.y;
            atomicOr(&taken[w][q >> 5], 1u << (q & 31));
          }
          const uint64_t sp = __ballot(spill);
          if (spill) spills[w][spilled + __popcll(sp & below)] = (uint16_t)p;
          spilled += __popcll(sp);
          m &= m - 1;
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    int free_before = 0;
    for (int q0 = 0; q0 < 8 * G * ((passes + 7) / 8); q0 += 64) {
      const int q = q0 + lane;
      const bool open = q < slots && !((taken[w][q >> 5] >> (q & 31)) & 1u);
      const uint64_t bal = __ballot(open);
      const int k = free_before + __popcll(bal & below);
      free_before += __popcll(bal);
      if (open || (q >= slots && q < 8 * G * ((passes + 7) / 8)))
        put(q / G, q % G, open && k < spilled ? (uint32_t)spills[w][k] : (uint32_t)(ul + a));
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

// rec[6 q .. 6 q + 2] = coordinates of slot q (zeros for a padding slot), rec[6 q + 3 ..] = 0. Flags bit 4: an x whose
// square overflows (the product's dummy records lie as far off).
__global__ void k_tile_coords(int64_t slots, const int32_t *__restrict__ tile_atoms, const double *__restrict__ xyz,
                              double *__restrict__ rec, int32_t *__restrict__ flags) {
  const int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (q >= slots) return;
  const int32_t at = tile_atoms[q];
  if (at >= 0 && !(fabs(xyz[3 * (int64_t)at]) < 1e150)) atomicOr(flags, 16);
  for (int k = 0; k < 3; ++k) {
    rec[6 * q + k] = at >= 0 ? xyz[3 * (int64_t)at + k] : 0.0;
    rec[6 * q + 3 + k] = 0.0;
  }
}

struct DevBuf {
  void *p = nullptr;
  ~DevBuf() {
    if (p) (void)hipFree(p);
  }
};

}  // namespace

// Out of device memory is INCH_ERR_CAPACITY (a caller may fall back on a form that needs less), and leaves no error
// behind for the next launch to report.
#define HIP_TRY(expr)                                                                      \
  do {                                                                                     \
    hipError_t _e = (expr);                                                                \
    if (_e == hipErrorOutOfMemory) (void)hipGetLastError();                                \
    if (_e != hipSuccess)                                                                  \
      INCH_FAIL(_e == hipErrorOutOfMemory ? INCH_ERR_CAPACITY : INCH_ERR_HIP, "%s: %s", #expr, hipGetErrorString(_e)); \
  } while (0)

namespace {

// out[0..m] = exclusive scan of in[0..m-1] (out[m] = total), on stream st; the tile
// temporaries are allocated here and freed after the scan has finished.
template <typename T>
inch_status scan_exclusive(int64_t m, const T *in, T *out, hipStream_t st) {
  const int64_t nt = scan_tiles(m);
  DevBuf sums, offs;
  if (nt > 4) {
    HIP_TRY(hipMalloc(&sums.p, (nt + 1) * sizeof(T)));
    HIP_TRY(hipMalloc(&offs.p, (nt + 1) * sizeof(T)));
  }
  HIP_TRY(scan_exclusive_into(m, in, out, (T *)sums.p, (T *)offs.p, st));
  if (nt > 4) HIP_TRY(hipStreamSynchronize(st));
  return INCH_OK;
}

}  // namespace

#define SCAN_TRY(m, in, out)                                   \
  do {                                                         \
    const inch_status _s = scan_exclusive((m), (in), (out), st); \
    if (_s != INCH_OK) return _s;                              \
  } while (0)

namespace {

// Scratch of the cell lists, cut from one allocation: cell of every atom, cell counts and starts,
// atoms and coordinates in cell order, row lengths, scan temporaries and the longest row.
struct CellWork {
  int32_t *cell_of, *cnt, *start, *atoms, *longest;
  int64_t *counts, *tsum, *toff;
  double *cx;
  int64_t bytes;
  CellWork(int64_t n, int64_t ncell, char *p) {
    const int64_t tiles = std::max(scan_tiles(ncell), scan_tiles(n)) + 2;
    int64_t at = 0;
    auto take = [&](int64_t b) {
      char *q = p + at;
      at += (b + 255) & ~(int64_t)255;
      return q;
    };
    cx = (double *)take(24 * n);
    counts = (int64_t *)take(8 * n);
    tsum = (int64_t *)take(8 * tiles);
    toff = (int64_t *)take(8 * tiles);
    cell_of = (int32_t *)take(4 * n);
    atoms = (int32_t *)take(4 * n);
    cnt = (int32_t *)take(4 * (ncell + 1));
    start = (int32_t *)take(4 * (ncell + 1));
    longest = (int32_t *)take(4);
    bytes = at;
  }
};

// grid: lo[3], 1 / cell size, dim[3] of cells of about the cutoff over the atoms' bounding box; part:
// device scratch of 256 x 6 doubles. Syncs.
inch_status cell_grid(int64_t n, const double *xyz, double rc, double *part, Grid &g, int64_t &ncell, const char *who,
                      hipStream_t st) {
  const int nb = 256;
  k_minmax<<<nb, 256, 0, st>>>(n, xyz, part);
  HIP_TRY(hipGetLastError());
  std::vector<double> hp(nb * 6);
  HIP_TRY(hipMemcpyAsync(hp.data(), part, nb * 6 * sizeof(double), hipMemcpyDeviceToHost, st));
  HIP_TRY(hipStreamSynchronize(st));
  double hi[3];
  for (int a = 0; a < 3; ++a) {
    g.lo[a] = INFINITY;
    hi[a] = -INFINITY;
    bool nan = false;   // std::min/max would drop a NaN partial
    for (int b = 0; b < nb; ++b) {
      nan |= std::isnan(hp[b * 6 + a]) || std::isnan(hp[b * 6 + 3 + a]);
      g.lo[a] = std::min(g.lo[a], hp[b * 6 + a]);
      hi[a] = std::max(hi[a], hp[b * 6 + 3 + a]);
    }
    if (nan || !std::isfinite(g.lo[a]) || !std::isfinite(hi[a])) INCH_FAIL(INCH_ERR_NAN, "%s: non-finite coordinates", who);
  }
  // cells a millionth wider than the cutoff: (v - lo) inv is off by at most 3 roundings, 4e-7 at 1.1e9 cells, so that
  // two atoms within the cutoff never lie two cells apart
  g.inv = (1.0 - 1e-6) / rc;
  ncell = 1;
  for (int a = 0; a < 3; ++a) {
    const double d = std::floor((hi[a] - g.lo[a]) * g.inv) + 1.0;
    // beyond what cells can be numbered by: one for all (cell_coord cuts there), as long as the other axes have few
    if (d >= 1.1e9 && d < 9.2e18) INCH_FAIL(INCH_ERR_CAPACITY, "%s: %g cells along one axis", who, d);
    g.dim[a] = d < 1.1e9 ? std::max<int64_t>(1, (int64_t)d) : 1;
    if (ncell > ((int64_t)1 << 30) / g.dim[a]) INCH_FAIL(INCH_ERR_CAPACITY, "%s: more than 2^30 cells", who);
    ncell *= g.dim[a];
  }
  return INCH_OK;
}

// The cell lists and, with indptr, the rows' lengths scanned into it.
inch_status cell_lists(int64_t n, const double *xyz, double rc, const Grid &g, int64_t ncell, const CellWork &k,
                       int64_t *indptr, hipStream_t st) {
  HIP_TRY(hipMemsetAsync(k.cnt, 0, (ncell + 1) * sizeof(int32_t), st));
  HIP_TRY(hipMemsetAsync(k.longest, 0, sizeof(int32_t), st));
  const int bs = 256;
  const unsigned gb = (unsigned)((n + bs - 1) / bs);
  k_cell_count<<<gb, bs, 0, st>>>(n, xyz, g, k.cell_of, k.cnt);
  HIP_TRY(hipGetLastError());
  HIP_TRY(scan_exclusive_into<int32_t>(ncell, k.cnt, k.start, (int32_t *)k.tsum, (int32_t *)k.toff, st));
  HIP_TRY(hipMemsetAsync(k.cnt, 0, (ncell + 1) * sizeof(int32_t), st));
  k_cell_fill<<<gb, bs, 0, st>>>(n, k.cell_of, k.start, k.cnt, k.atoms);
  k_cell_coords<<<(unsigned)((3 * n + bs - 1) / bs), bs, 0, st>>>(n, xyz, k.atoms, k.cx);
  HIP_TRY(hipGetLastError());
  if (!indptr) return INCH_OK;
  k_neigh<false><<<(unsigned)((n + kRun - 1) / kRun), 256, 0, st>>>(n, g, rc * rc, k.start, k.atoms, k.cx, nullptr,
                                                                    k.counts, k.longest, nullptr);
  HIP_TRY(hipGetLastError());
  HIP_TRY(scan_exclusive_into<int64_t>(n, k.counts, indptr, k.tsum, k.toff, st));
  return INCH_OK;
}

inch_status cell_fill(int64_t n, double rc, const Grid &g, const CellWork &k, const int64_t *indptr, int32_t *indices,
                      hipStream_t st) {
  k_neigh<true><<<(unsigned)((n + kRun - 1) / kRun), 256, 0, st>>>(n, g, rc * rc, k.start, k.atoms, k.cx, indptr,
                                                                   nullptr, nullptr, indices);
  HIP_TRY(hipGetLastError());
  return INCH_OK;
}

void grid_to_plan(const Grid &g, double *plan) {
  for (int a = 0; a < 3; ++a) {
    plan[a] = g.lo[a];
    plan[4 + a] = (double)g.dim[a];
  }
  plan[3] = g.inv;
}

Grid plan_to_grid(const double *plan, int64_t &ncell) {
  Grid g;
  ncell = 1;
  for (int a = 0; a < 3; ++a) {
    g.lo[a] = plan[a];
    g.dim[a] = (int64_t)plan[4 + a];
    ncell *= g.dim[a];
  }
  g.inv = plan[3];
  return g;
}

}  // namespace

extern "C" inch_status inch_cells_plan(int64_t n, const double *xyz, double rc, double *plan, int64_t *work_bytes,
                                       double *scratch, void *stream) {
  INCH_REQUIRE(n > 0 && xyz && rc > 0 && plan && work_bytes && scratch, "inch_cells_plan: bad args");
  INCH_REQUIRE(n < (int64_t)1 << 31, "inch_cells_plan: n must fit int32");
  Grid g;
  int64_t ncell = 0;
  const inch_status s = cell_grid(n, xyz, rc, scratch, g, ncell, "inch_neighbors_celllist", (hipStream_t)stream);
  if (s != INCH_OK) return s;
  grid_to_plan(g, plan);
  *work_bytes = CellWork(n, ncell, nullptr).bytes;
  return INCH_OK;
}

extern "C" inch_status inch_cells_count(int64_t n, const double *xyz, double rc, const double *plan, void *work,
                                        int64_t work_bytes, int64_t *indptr, int64_t *nnz_out, void *stream) {
  INCH_REQUIRE(n > 0 && xyz && rc > 0 && plan && work && indptr && nnz_out, "inch_cells_count: bad args");
  int64_t ncell = 0;
  const Grid g = plan_to_grid(plan, ncell);
  const CellWork k(n, ncell, (char *)work);
  INCH_REQUIRE(work_bytes >= k.bytes, "inch_cells_count: work too small");
  hipStream_t st = (hipStream_t)stream;
  const inch_status s = cell_lists(n, xyz, rc, g, ncell, k, indptr, st);
  if (s != INCH_OK) return s;
  int32_t longest = 0;
  HIP_TRY(hipMemcpyAsync(&longest, k.longest, sizeof(longest), hipMemcpyDeviceToHost, st));
  HIP_TRY(hipMemcpyAsync(nnz_out, indptr + n, sizeof(int64_t), hipMemcpyDeviceToHost, st));
  HIP_TRY(hipStreamSynchronize(st));
  if (longest > kMaxRow) INCH_FAIL(INCH_ERR_CAPACITY, "inch_neighbors_celllist: a row has %d neighbours (> %d)", longest, kMaxRow);
  return INCH_OK;
}

extern "C" inch_status inch_cells_fill(int64_t n, double rc, const double *plan, void *work, int64_t work_bytes,
                                       const int64_t *indptr, int32_t *indices, int32_t sorted, void *stream) {
  INCH_REQUIRE(n > 0 && rc > 0 && plan && work && indptr && indices, "inch_cells_fill: bad args");
  int64_t ncell = 0;
  const Grid g = plan_to_grid(plan, ncell);
  const CellWork k(n, ncell, (char *)work);
  INCH_REQUIRE(work_bytes >= k.bytes, "inch_cells_fill: work too small");
  hipStream_t st = (hipStream_t)stream;
  const inch_status s = cell_fill(n, rc, g, k, indptr, indices, st);
  if (s != INCH_OK || !sorted) return s;
  k_sort_rows<<<(unsigned)n, 64, 0, st>>>(n, indptr, indices, k.longest);
  HIP_TRY(hipGetLastError());
  return INCH_OK;
}

extern "C" inch_status inch_neighbors_celllist(int64_t n, const double *xyz, double rc, int64_t *indptr,
                                               int32_t *indices, int64_t capacity, int64_t *nnz_out,
                                               void *stream) {
  INCH_REQUIRE(n > 0 && xyz && indptr && rc > 0, "inch_neighbors_celllist: bad args");
  INCH_REQUIRE(n < (int64_t)1 << 31, "inch_neighbors_celllist: n must fit int32");
  hipStream_t st = (hipStream_t)stream;
  DevBuf part, work;
  HIP_TRY(hipMalloc(&part.p, 256 * 6 * sizeof(double)));
  Grid g;
  int64_t ncell = 0;
  inch_status s = cell_grid(n, xyz, rc, (double *)part.p, g, ncell, "inch_neighbors_celllist", st);
  if (s != INCH_OK) return s;
  HIP_TRY(hipMalloc(&work.p, CellWork(n, ncell, nullptr).bytes));
  const CellWork k(n, ncell, (char *)work.p);
  s = cell_lists(n, xyz, rc, g, ncell, k, indices ? nullptr : indptr, st);
  if (s != INCH_OK) return s;
  int64_t total = 0;
  HIP_TRY(hipMemcpyAsync(&total, indptr + n, sizeof(int64_t), hipMemcpyDeviceToHost, st));
  HIP_TRY(hipStreamSynchronize(st));
  if (indices) {
    if (total > capacity) INCH_FAIL(INCH_ERR_CAPACITY, "inch_neighbors_celllist: need %lld > capacity %lld", (long long)total, (long long)capacity);
    s = cell_fill(n, rc, g, k, indptr, indices, st);
    if (s != INCH_OK) return s;
    k_sort_rows<<<(unsigned)n, 64, 0, st>>>(n, indptr, indices, k.longest);
    HIP_TRY(hipGetLastError());
    int32_t over = 0;
    HIP_TRY(hipMemcpyAsync(&over, k.longest, sizeof(int32_t), hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    if (over) INCH_FAIL(INCH_ERR_CAPACITY, "inch_neighbors_celllist: a row has %d neighbours (> %d)", over, kMaxRow);
  }
  if (nnz_out) *nnz_out = total;
  return INCH_OK;
}

extern "C" inch_status inch_csr_permute(int64_t n, const int64_t *indptr, const int32_t *indices,
                                        const int32_t *order, const int64_t *undo, int64_t *out_indptr,
                                        int32_t *out_indices, void *stream) {
  INCH_REQUIRE(n > 0 && indptr && indices && order && undo && out_indptr && out_indices, "inch_csr_permute: bad args");
  hipStream_t st = (hipStream_t)stream;
  DevBuf counts, ovf;
  HIP_TRY(hipMalloc(&counts.p, n * sizeof(int64_t)));
  HIP_TRY(hipMalloc(&ovf.p, sizeof(int32_t)));
  HIP_TRY(hipMemsetAsync(ovf.p, 0, sizeof(int32_t), st));
  const int bs = 256;
  k_perm_counts<<<(unsigned)((n + bs - 1) / bs), bs, 0, st>>>(n, indptr, order, (int64_t *)counts.p);
  HIP_TRY(hipGetLastError());
  SCAN_TRY(n, (const int64_t *)counts.p, out_indptr);
  k_permute_sort_rows<<<(unsigned)n, 64, 0, st>>>(n, indptr, indices, order, undo, out_indptr, out_indices,
                                                  (int32_t *)ovf.p);
  HIP_TRY(hipGetLastError());
  int32_t over = 0;
  HIP_TRY(hipMemcpyAsync(&over, ovf.p, sizeof(int32_t), hipMemcpyDeviceToHost, st));
  HIP_TRY(hipStreamSynchronize(st));
  if (over) INCH_FAIL(INCH_ERR_CAPACITY, "inch_csr_permute: a row has %d entries (> %d)", over, kMaxRow);
  return INCH_OK;
}

extern "C" inch_status inch_hessian_assemble(int64_t n, const double *xyz, double rc, double plus_i,
                                             const int64_t *rowptr, const int32_t *col, double *vals64,
                                             float *vals32, double *diag, void *stream) {
  (void)rc;  // the pattern already encodes the cutoff; only r^2 == 0 is masked here
  INCH_REQUIRE(n > 0 && xyz && rowptr && col, "inch_hessian_assemble: bad args");
  INCH_REQUIRE(vals64 || vals32 || diag, "inch_hessian_assemble: no output");
  hipStream_t st = (hipStream_t)stream;
  const int bs = 256;
  const int64_t grid = (n * 64 + bs - 1) / bs;
  k_assemble<<<grid, bs, 0, st>>>(n, xyz, plus_i, rowptr, col, nullptr, 0.0, 0.0, vals64, vals32, diag);
  HIP_TRY(hipGetLastError());
  return INCH_OK;
}

extern "C" inch_status inch_neighbors_celllist_pbc(int64_t n, const double *xyz, double rc, double box_x,
                                                   double box_y, double origin_x, double origin_y, int64_t *indptr,
                                                   int32_t *indices, uint16_t *images, int64_t capacity,
                                                   int64_t *nnz_out, void *stream) {
  INCH_REQUIRE(n > 0 && xyz && indptr && rc > 0, "inch_neighbors_celllist_pbc: bad args");
  INCH_REQUIRE(box_x > rc && box_y > rc, "ABORTED. The PBC box size must exceed the cutoff (%g, %g vs %g)", box_x,
               box_y, rc);
  INCH_REQUIRE(n < (int64_t)1 << 31, "inch_neighbors_celllist_pbc: n must fit int32");
  INCH_REQUIRE(!indices || images, "inch_neighbors_celllist_pbc: the fill pass needs images");
  hipStream_t st = (hipStream_t)stream;
  const int nb = 256;
  DevBuf part;
  HIP_TRY(hipMalloc(&part.p, nb * 6 * sizeof(double)));
  k_minmax<<<nb, 256, 0, st>>>(n, xyz, (double *)part.p);
  HIP_TRY(hipGetLastError());
  std::vector<double> hp(nb * 6);
  HIP_TRY(hipMemcpyAsync(hp.data(), part.p, nb * 6 * sizeof(double), hipMemcpyDeviceToHost, st));
  HIP_TRY(hipStreamSynchronize(st));
  double zlo = INFINITY, zhi = -INFINITY;
  for (int b = 0; b < nb; ++b) {
    for (int a = 0; a < 3; ++a)
      if (!std::isfinite(hp[b * 6 + a]) && hp[b * 6 + a] != INFINITY)
        INCH_FAIL(INCH_ERR_NAN, "inch_neighbors_celllist_pbc: non-finite coordinates");
    zlo = std::min(zlo, hp[b * 6 + 2]);
    zhi = std::max(zhi, hp[b * 6 + 5]);
  }
  if (!std::isfinite(zlo) || !std::isfinite(zhi)) INCH_FAIL(INCH_ERR_NAN, "inch_neighbors_celllist_pbc: non-finite coordinates");
  PbcGrid g;
  g.lo[0] = origin_x;
  g.lo[1] = origin_y;
  g.lo[2] = zlo;
  g.box[0] = box_x;
  g.box[1] = box_y;
  g.dim[0] = std::max<int64_t>(1, (int64_t)std::floor(box_x / rc));
  g.dim[1] = std::max<int64_t>(1, (int64_t)std::floor(box_y / rc));
  g.cell[0] = box_x / (double)g.dim[0];
  g.cell[1] = box_y / (double)g.dim[1];
  g.cell[2] = rc;
  g.dim[2] = std::max<int64_t>(1, (int64_t)std::floor((zhi - zlo) / rc) + 1);
  const int64_t ncell = g.dim[0] * g.dim[1] * g.dim[2];
  if (ncell > ((int64_t)1 << 30)) INCH_FAIL(INCH_ERR_CAPACITY, "inch_neighbors_celllist_pbc: %lld cells", (long long)ncell);
  DevBuf cell_of, cnt, start, atoms, counts, ovf;
  HIP_TRY(hipMalloc(&cell_of.p, n * sizeof(int32_t)));
  HIP_TRY(hipMalloc(&cnt.p, (ncell + 1) * sizeof(int32_t)));
  HIP_TRY(hipMalloc(&start.p, (ncell + 1) * sizeof(int32_t)));
  HIP_TRY(hipMalloc(&atoms.p, n * sizeof(int32_t)));
  HIP_TRY(hipMemsetAsync(cnt.p, 0, (ncell + 1) * sizeof(int32_t), st));
  const int bs = 256;
  const int64_t gb = (n + bs - 1) / bs;
  k_cell_count_pbc<<<gb, bs, 0, st>>>(n, xyz, g, (int32_t *)cell_of.p, (int32_t *)cnt.p);
  HIP_TRY(hipGetLastError());
  SCAN_TRY(ncell, (const int32_t *)cnt.p, (int32_t *)start.p);
  HIP_TRY(hipMemsetAsync(cnt.p, 0, (ncell + 1) * sizeof(int32_t), st));
  k_cell_fill<<<gb, bs, 0, st>>>(n, (int32_t *)cell_of.p, (int32_t *)start.p, (int32_t *)cnt.p, (int32_t *)atoms.p);
  HIP_TRY(hipGetLastError());
  const double rc2 = rc * rc;
  if (indices == nullptr) {
    HIP_TRY(hipMalloc(&counts.p, n * sizeof(int64_t)));
    k_neigh_pbc<<<gb, bs, 0, st>>>(n, xyz, g, rc2, (int32_t *)start.p, (int32_t *)atoms.p, nullptr,
                                   (int64_t *)counts.p, nullptr);
    HIP_TRY(hipGetLastError());
    SCAN_TRY(n, (const int64_t *)counts.p, indptr);
    int64_t total = 0;
    HIP_TRY(hipMemcpyAsync(&total, indptr + n, sizeof(int64_t), hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    if (nnz_out) *nnz_out = total;
    return INCH_OK;
  }
  int64_t total = 0;
  HIP_TRY(hipMemcpyAsync(&total, indptr + n, sizeof(int64_t), hipMemcpyDeviceToHost, st));
  HIP_TRY(hipStreamSynchronize(st));
  if (total > capacity) INCH_FAIL(INCH_ERR_CAPACITY, "inch_neighbors_celllist_pbc: need %lld > capacity %lld", (long long)total, (long long)capacity);
  k_neigh_pbc<<<gb, bs, 0, st>>>(n, xyz, g, rc2, (int32_t *)start.p, (int32_t *)atoms.p, indptr, nullptr, indices);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipMalloc(&ovf.p, sizeof(int32_t)));
  HIP_TRY(hipMemsetAsync(ovf.p, 0, sizeof(int32_t), st));
  k_sort_rows<<<n, 64, 0, st>>>(n, indptr, indices, (int32_t *)ovf.p);
  HIP_TRY(hipGetLastError());
  int32_t over = 0;
  HIP_TRY(hipMemcpyAsync(&over, ovf.p, sizeof(int32_t), hipMemcpyDeviceToHost, st));
  HIP_TRY(hipStreamSynchronize(st));
  if (over) INCH_FAIL(INCH_ERR_CAPACITY, "inch_neighbors_celllist_pbc: a row has %d neighbours (> %d)", over, kMaxRow);
  k_image_masks<<<gb, bs, 0, st>>>(n, xyz, box_x, box_y, rc2, indptr, indices, images);
  HIP_TRY(hipGetLastError());
  if (nnz_out) *nnz_out = total;
  return INCH_OK;
}

extern "C" inch_status inch_hessian_assemble_pbc(int64_t n, const double *xyz, double plus_i, const int64_t *rowptr,
                                                 const int32_t *col, const uint16_t *images, double box_x,
                                                 double box_y, double *vals64, float *vals32, double *diag,
                                                 void *stream) {
  INCH_REQUIRE(n > 0 && xyz && rowptr && col && images && box_x > 0 && box_y > 0, "inch_hessian_assemble_pbc: bad args");
  INCH_REQUIRE(vals64 || vals32 || diag, "inch_hessian_assemble_pbc: no output");
  hipStream_t st = (hipStream_t)stream;
  const int bs = 256;
  const int64_t grid = (n * 64 + bs - 1) / bs;
  k_assemble<<<grid, bs, 0, st>>>(n, xyz, plus_i, rowptr, col, images, box_x, box_y, vals64, vals32, diag);
  HIP_TRY(hipGetLastError());
  return INCH_OK;
}

// The cluster layout, in two calls (one_pass = false: the first, without entries, builds the
// clusters and their counts; the second, with entries, merges the rows again in the final
// numbering) or in one (the count pass also writes each list into a provisional buffer with
// room for the cluster's row entries, and the lists are copied into the final numbering).
static inch_status anm_clusters_impl(int64_t n, const double *xyz, const int64_t *rowptr, const int32_t *col,
                                     double cell_xy, double cell_z, int32_t *cluster_atoms, int64_t *cl_ptr,
                                     int32_t *base, uint32_t *entries, int64_t capacity, int64_t *nnz_out,
                                     void *stream, bool one_pass) {
  INCH_REQUIRE(n > 0 && xyz && rowptr && col && cluster_atoms && cl_ptr && base && cell_xy > 0 && cell_z > 0,
               "inch_anm_clusters: bad args");
  INCH_REQUIRE(n < (int64_t)1 << 31, "inch_anm_clusters: n must fit int32");
  // the cluster kernels address coordinates and vectors with 32-bit byte offsets
  if (24 * n > (int64_t)UINT32_MAX) INCH_FAIL(INCH_ERR_CAPACITY, "inch_anm_clusters: n = %lld exceeds the 32-bit offset range (%lld atoms)", (long long)n, (long long)(UINT32_MAX / 24));
  hipStream_t st = (hipStream_t)stream;
  const int64_t ncl = (n + kClusterAtoms - 1) / kClusterAtoms;
  DevBuf ovf;
  HIP_TRY(hipMalloc(&ovf.p, sizeof(int32_t)));
  HIP_TRY(hipMemsetAsync(ovf.p, 0, sizeof(int32_t), st));
  auto check_overflow = [&](const char *pass) -> inch_status {
    int32_t over = 0;
    HIP_TRY(hipMemcpyAsync(&over, ovf.p, sizeof(int32_t), hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    if (over & 1) INCH_FAIL(INCH_ERR_CAPACITY, "inch_anm_clusters (%s): a cluster's rows hold more than %d entries", pass, kMaxUnion);
    if (over & 2) INCH_FAIL(INCH_ERR_CAPACITY, "inch_anm_clusters (%s): a cluster's neighbours span 2^24 columns or more", pass);
    if (over & 4) INCH_FAIL(INCH_ERR_INVALID, "inch_anm_clusters (%s): a row's columns are not in ascending order or outside [0, n)", pass);
    return INCH_OK;
  };
  if (entries && !one_pass) {  // fill pass on the layout of the count pass
    int64_t total = 0;
    HIP_TRY(hipMemcpyAsync(&total, cl_ptr + ncl, sizeof(int64_t), hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    if (total > capacity) INCH_FAIL(INCH_ERR_CAPACITY, "inch_anm_clusters: need %lld > capacity %lld", (long long)total, (long long)capacity);
    k_cl_union<true><<<(unsigned)ncl, 256, 0, st>>>(n, ncl, xyz, rowptr, col, cluster_atoms, cl_ptr, base, nullptr, entries,
                                                    (int32_t *)ovf.p);
    HIP_TRY(hipGetLastError());
    inch_status s = check_overflow("fill");
    if (s != INCH_OK) return s;
    if (nnz_out) *nnz_out = total;
    return INCH_OK;
  }
  // bounds
  const int nb = 256;
  DevBuf part;
  HIP_TRY(hipMalloc(&part.p, nb * 6 * sizeof(double)));
  k_minmax<<<nb, 256, 0, st>>>(n, xyz, (double *)part.p);
  HIP_TRY(hipGetLastError());
  std::vector<double> hp(nb * 6);
  HIP_TRY(hipMemcpyAsync(hp.data(), part.p, nb * 6 * sizeof(double), hipMemcpyDeviceToHost, st));
  HIP_TRY(hipStreamSynchronize(st));
  CGrid g;
  double hi[3];
  for (int a = 0; a < 3; ++a) {
    g.lo[a] = INFINITY;
    hi[a] = -INFINITY;
    bool nan = false;   // std::min/max would drop a NaN partial
    for (int b = 0; b < nb; ++b) {
      nan |= std::isnan(hp[b * 6 + a]) || std::isnan(hp[b * 6 + 3 + a]);
      g.lo[a] = std::min(g.lo[a], hp[b * 6 + a]);
      hi[a] = std::max(hi[a], hp[b * 6 + 3 + a]);
    }
    if (nan || !std::isfinite(g.lo[a]) || !std::isfinite(hi[a])) INCH_FAIL(INCH_ERR_NAN, "inch_anm_clusters: non-finite coordinates");
  }
  // cells: cell_xy in x and y; cell_z in z, coarsened only beyond max(16n, 65536) cells (an
  // assembly's bounding box is mostly empty: coarser cells would make its clusters taller)
  const double size[3] = {cell_xy, cell_xy, cell_z};
  for (int a = 0; a < 3; ++a) {
    g.inv[a] = 1.0 / size[a];
    g.dim[a] = std::max<int64_t>(1, (int64_t)std::floor((hi[a] - g.lo[a]) * g.inv[a]) + 1);
  }
  const int64_t cap_cells = std::max<int64_t>(16 * n, 65536);
  while (g.dim[0] * g.dim[1] * g.dim[2] > cap_cells && g.dim[2] > 1) {
    g.inv[2] *= 0.5;
    g.dim[2] = std::max<int64_t>(1, (int64_t)std::floor((hi[2] - g.lo[2]) * g.inv[2]) + 1);
  }
  const int64_t ncell = g.dim[0] * g.dim[1] * g.dim[2];
  if (ncell > ((int64_t)1 << 30)) INCH_FAIL(INCH_ERR_CAPACITY, "inch_anm_clusters: %lld cells", (long long)ncell);
  DevBuf cell_of, cnt, start, atoms, counts;
  HIP_TRY(hipMalloc(&cell_of.p, n * sizeof(int32_t)));
  HIP_TRY(hipMalloc(&cnt.p, (ncell + 1) * sizeof(int32_t)));
  HIP_TRY(hipMalloc(&start.p, (ncell + 1) * sizeof(int32_t)));
  HIP_TRY(hipMalloc(&atoms.p, n * sizeof(int32_t)));
  HIP_TRY(hipMalloc(&counts.p, ncl * sizeof(int64_t)));
  HIP_TRY(hipMemsetAsync(cnt.p, 0, (ncell + 1) * sizeof(int32_t), st));
  const int bs = 256;
  const int64_t gb = (n + bs - 1) / bs;
  k_cl_cell<<<gb, bs, 0, st>>>(n, xyz, g, (int32_t *)cell_of.p, (int32_t *)cnt.p);
  HIP_TRY(hipGetLastError());
  SCAN_TRY(ncell, (const int32_t *)cnt.p, (int32_t *)start.p);
  HIP_TRY(hipMemsetAsync(cnt.p, 0, (ncell + 1) * sizeof(int32_t), st));
  k_cell_fill<<<gb, bs, 0, st>>>(n, (int32_t *)cell_of.p, (int32_t *)start.p, (int32_t *)cnt.p, (int32_t *)atoms.p);
  HIP_TRY(hipGetLastError());
  k_cell_isort<<<(unsigned)((ncell + bs - 1) / bs), bs, 0, st>>>(ncell, (int32_t *)start.p, (int32_t *)atoms.p);
  HIP_TRY(hipGetLastError());
  const int64_t slots = ncl * kClusterAtoms;
  k_cl_atoms<<<(unsigned)((slots + bs - 1) / bs), bs, 0, st>>>(n, slots, (int32_t *)atoms.p, cluster_atoms);
  HIP_TRY(hipGetLastError());
  DevBuf atoms0, counts0, base0, perm;
  HIP_TRY(hipMalloc(&atoms0.p, slots * sizeof(int32_t)));
  HIP_TRY(hipMalloc(&counts0.p, ncl * sizeof(int64_t)));
  HIP_TRY(hipMalloc(&base0.p, ncl * sizeof(int32_t)));
  HIP_TRY(hipMalloc(&perm.p, ncl * sizeof(uint64_t)));
  HIP_TRY(hipMemcpyAsync(atoms0.p, cluster_atoms, slots * sizeof(int32_t), hipMemcpyDeviceToDevice, st));
  DevBuf prov_ptr, prov;
  if (one_pass) {   // room for every cluster's row entries, in the count pass's numbering
    HIP_TRY(hipMalloc(&prov_ptr.p, (ncl + 1) * sizeof(int64_t)));
    k_cl_totals<<<(unsigned)((ncl + bs - 1) / bs), bs, 0, st>>>(ncl, (int32_t *)atoms0.p, rowptr,
                                                               (int64_t *)counts0.p);
    HIP_TRY(hipGetLastError());
    SCAN_TRY(ncl, (const int64_t *)counts0.p, (int64_t *)prov_ptr.p);
    int64_t room = 0;
    HIP_TRY(hipMemcpyAsync(&room, (int64_t *)prov_ptr.p + ncl, sizeof(int64_t), hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    HIP_TRY(hipMalloc(&prov.p, std::max<int64_t>(1, room) * sizeof(uint32_t)));
  }
  k_cl_union<false><<<(unsigned)ncl, 256, 0, st>>>(n, ncl, xyz, rowptr, col, (int32_t *)atoms0.p, nullptr, (int32_t *)base0.p,
                                                   (int64_t *)counts0.p, (uint32_t *)prov.p, (int32_t *)ovf.p,
                                                   (const int64_t *)prov_ptr.p);
  HIP_TRY(hipGetLastError());
  {
    inch_status s0 = check_overflow("count");
    if (s0 != INCH_OK) return s0;
  }
  // clusters in the order of their smallest neighbour (ties by spatial order): consecutive
  // clusters, and so each XCD's contiguous share of them, gather from one band of the
  // vectors, which are in the matrix's (RCM) order. Radix sort of the keys on the device.
  DevBuf keys, tmp;
  HIP_TRY(hipMalloc(&keys.p, ncl * sizeof(uint64_t)));
  k_cl_keys<<<(unsigned)((ncl + bs - 1) / bs), bs, 0, st>>>(ncl, (int32_t *)base0.p, (uint64_t *)keys.p);
  HIP_TRY(hipGetLastError());
  size_t tmp_bytes = 0;
  HIP_TRY(hipcub::DeviceRadixSort::SortKeys(nullptr, tmp_bytes, (const uint64_t *)keys.p, (uint64_t *)perm.p,
                                            (int)ncl, 0, 64, st));
  HIP_TRY(hipMalloc(&tmp.p, tmp_bytes));
  HIP_TRY(hipcub::DeviceRadixSort::SortKeys(tmp.p, tmp_bytes, (const uint64_t *)keys.p, (uint64_t *)perm.p, (int)ncl,
                                            0, 64, st));
  k_cl_permute<<<(unsigned)((ncl + bs - 1) / bs), bs, 0, st>>>(ncl, (const uint64_t *)perm.p, (int32_t *)atoms0.p,
                                                              (int64_t *)counts0.p, (int32_t *)base0.p, cluster_atoms,
                                                              (int64_t *)counts.p, base);
  HIP_TRY(hipGetLastError());
  SCAN_TRY(ncl, (const int64_t *)counts.p, cl_ptr);
  inch_status s = check_overflow("count");
  if (s != INCH_OK) return s;
  int64_t total = 0;
  HIP_TRY(hipMemcpyAsync(&total, cl_ptr + ncl, sizeof(int64_t), hipMemcpyDeviceToHost, st));
  HIP_TRY(hipStreamSynchronize(st));
  if (nnz_out) *nnz_out = total;
  if (one_pass) {
    if (total > capacity) INCH_FAIL(INCH_ERR_CAPACITY, "inch_anm_clusters_one_pass: need %lld > capacity %lld", (long long)total, (long long)capacity);
    k_cl_copy<<<(unsigned)ncl, 256, 0, st>>>(ncl, (const uint64_t *)perm.p, (const int64_t *)prov_ptr.p,
                                             (const uint32_t *)prov.p, cl_ptr, entries);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(st));   // prov is freed on return
  }
  return INCH_OK;
}

extern "C" inch_status inch_anm_clusters(int64_t n, const double *xyz, const int64_t *rowptr, const int32_t *col,
                                         double cell_xy, double cell_z, int32_t *cluster_atoms, int64_t *cl_ptr,
                                         int32_t *base, uint32_t *entries, int64_t capacity, int64_t *nnz_out,
                                         void *stream) {
  return anm_clusters_impl(n, xyz, rowptr, col, cell_xy, cell_z, cluster_atoms, cl_ptr, base, entries, capacity,
                           nnz_out, stream, false);
}

extern "C" inch_status inch_anm_clusters_one_pass(int64_t n, const double *xyz, const int64_t *rowptr,
                                                  const int32_t *col, double cell_xy, double cell_z,
                                                  int32_t *cluster_atoms, int64_t *cl_ptr, int32_t *base,
                                                  uint32_t *entries, int64_t capacity, int64_t *nnz_out,
                                                  void *stream) {
  INCH_REQUIRE(entries && capacity >= 0, "inch_anm_clusters_one_pass: entries needed");
  return anm_clusters_impl(n, xyz, rowptr, col, cell_xy, cell_z, cluster_atoms, cl_ptr, base, entries, capacity,
                           nnz_out, stream, true);
}

extern "C" inch_status inch_anm_records(int64_t n, const double *xyz, int64_t ncl, const int32_t *cluster_atoms,
                                        const int64_t *cl_ptr, const int32_t *base, const uint32_t *entries,
                                        double *rec, uint32_t *rec_entries, void *stream) {
  INCH_REQUIRE(n > 0 && xyz && cluster_atoms && cl_ptr && base && entries && rec && rec_entries,
               "inch_anm_records: bad args");
  INCH_REQUIRE(ncl == (n + kClusterAtoms - 1) / kClusterAtoms, "inch_anm_records: ncl must be ceil(n / 4)");
  // the record product addresses records with 32-bit byte offsets (48 bytes per slot)
  if (192 * ncl > (int64_t)UINT32_MAX)
    INCH_FAIL(INCH_ERR_CAPACITY, "inch_anm_records: %lld clusters exceed the 32-bit record offsets", (long long)ncl);
  hipStream_t st = (hipStream_t)stream;
  const int64_t slots = kClusterAtoms * ncl;
  DevBuf slot_of;
  HIP_TRY(hipMalloc(&slot_of.p, n * sizeof(int32_t)));
  k_rec_coords<<<(unsigned)((slots + 255) / 256), 256, 0, st>>>(slots, cluster_atoms, xyz, rec, (int32_t *)slot_of.p);
  HIP_TRY(hipGetLastError());
  k_rec_lists<<<(unsigned)ncl, 256, 0, st>>>(ncl, cl_ptr, base, entries, (const int32_t *)slot_of.p, rec_entries);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(st));   // slot_of is freed on return
  return INCH_OK;
}

namespace {

constexpr int kBsrTileWords = 8192;   // 262,144 columns from the smallest to the largest of a tile's rows

// A workgroup per tile of rows order[start[t]] ..: the columns its rows name, each once and ascending, as set bits
// from the smallest column on. Their number goes to *umax (0x7fffffff when their span exceeds the bits) and ulen[t];
// with FILL ulist[t ustride ..] are these columns, uidx[b] the place of col[b] among them, and per place of the tile
// slots: its row (-1: none), the row's length and first block (low and high half). LDS atomics and one
// scan bound it; the lists of 150,000 atoms, their order and both passes take 0.9 ms.
template <bool FILL>
__global__ void __launch_bounds__(256) k_bsr_tiles(const int64_t *__restrict__ rowptr, const int32_t *__restrict__ col,
                                                    const int32_t *__restrict__ order,
                                                    const int32_t *__restrict__ start, int ustride,
                                                    int tile, int32_t *__restrict__ slots,
                                                    int32_t *__restrict__ ulen, int32_t *__restrict__ ulist,
                                                    uint16_t *__restrict__ uidx, int32_t *__restrict__ umax) {
  __shared__ uint32_t bits[kBsrTileWords];
  __shared__ uint16_t before[kBsrTileWords];
  __shared__ int32_t lo, hi, sums[256];
  const int t = blockIdx.x, tid = threadIdx.x;
  const int r0 = start[t], r1 = start[t + 1];
  if (tid == 0) {
    lo = 0x7fffffff;
    hi = -1;
  }
  __syncthreads();
  // a row per wave, its blocks over the lanes
  const int lane = tid & 63, w = tid >> 6;
  int mn = 0x7fffffff, mx = -1;
  for (int r = r0 + w; r < r1; r += 4)
    for (int64_t b = rowptr[order[r]] + lane; b < rowptr[order[r] + 1]; b += 64) {
      mn = min(mn, col[b]);
      mx = max(mx, col[b]);
    }
  atomicMin(&lo, mn);
  atomicMax(&hi, mx);
  __syncthreads();
  const int c0 = lo, words = hi < c0 ? 0 : ((hi - c0) >> 5) + 1;
  if (words > kBsrTileWords) {   // the same for all threads
    if (tid == 0) atomicMax(umax, 0x7fffffff);
    return;
  }
  for (int i = tid; i < words; i += 256) bits[i] = 0;
  __syncthreads();
  for (int r = r0 + w; r < r1; r += 4)
    for (int64_t b = rowptr[order[r]] + lane; b < rowptr[order[r] + 1]; b += 64) {
      const int d = col[b] - c0;
      atomicOr(&bits[d >> 5], 1u << (d & 31));
    }
  __syncthreads();
  // thread t takes words [t per, (t + 1) per)
  const int per = (words + 255) / 256, w0 = min(tid * per, words), w1 = min(w0 + per, words);
  int mine = 0;
  for (int i = w0; i < w1; ++i) mine += __popc(bits[i]);
  sums[tid] = mine;
  __syncthreads();
  for (int off = 1; off < 256; off <<= 1) {
    const int v = tid >= off ? sums[tid - off] : 0;
    __syncthreads();
    sums[tid] += v;
    __syncthreads();
  }
  const int total = sums[255];
  if (tid == 0) atomicMax(umax, total);
  if constexpr (!FILL) {
    if (tid == 0) ulen[t] = total;
    return;
  }
  if (total > ustride) return;   // the caller's stride is of other rows: refused by *umax
  if (tid < tile) {
    const int row = r0 + tid < r1 ? order[r0 + tid] : -1;
    const int32_t len = row < 0 ? 0 : (int32_t)(rowptr[row + 1] - rowptr[row]);
    const int64_t b = len > 0 ? rowptr[row] : 0;   // a place without blocks names block 0, which the product may read
    int32_t *q = slots + 4 * ((int64_t)t * tile + tid);
    q[0] = row;
    q[1] = len;
    q[2] = (int32_t)(uint32_t)b;
    q[3] = (int32_t)(b >> 32);
  }
  int at = sums[tid] - mine;
  for (int i = w0; i < w1; ++i) {
    before[i] = (uint16_t)at;
    for (uint32_t m = bits[i]; m; m &= m - 1) {
      ulist[(int64_t)t * ustride + at] = c0 + 32 * i + __ffs(m) - 1;
      ++at;
    }
  }
  __syncthreads();
  for (int r = r0 + w; r < r1; r += 4)
    for (int64_t b = rowptr[order[r]] + lane; b < rowptr[order[r] + 1]; b += 64) {
      const int d = col[b] - c0;
      uidx[b] = (uint16_t)(before[d >> 5] + __popc(bits[d >> 5] & ((1u << (d & 31)) - 1)));
    }
}

}  // namespace

extern "C" inch_status inch_bsr_tiles(int64_t n, const int64_t *rowptr, const int32_t *col, int64_t ntile,
                                      const int32_t *order, const int32_t *tile_start, int32_t tile, int32_t ustride,
                                      int32_t *slots, int32_t *ulen, int32_t *ulist, uint16_t *uidx, int32_t *umax_out,
                                      void *stream) {
  INCH_REQUIRE(n > 0 && n < (int64_t)1 << 31 && rowptr && col && ntile > 0 && ntile <= n && order && tile_start && ulen,
               "inch_bsr_tiles: bad args");
  INCH_REQUIRE(ulist ? slots && uidx && tile > 0 && tile <= 256 && ustride > 0 && ustride <= 65536 : umax_out != nullptr,
               "inch_bsr_tiles: bad lists");
  hipStream_t st = (hipStream_t)stream;
  DevBuf um;
  HIP_TRY(hipMalloc(&um.p, sizeof(int32_t)));
  HIP_TRY(hipMemsetAsync(um.p, 0, sizeof(int32_t), st));
  if (ulist)
    k_bsr_tiles<true><<<(unsigned)ntile, 256, 0, st>>>(rowptr, col, order, tile_start, ustride, tile, slots, ulen, ulist,
                                                       uidx, (int32_t *)um.p);
  else
    k_bsr_tiles<false><<<(unsigned)ntile, 256, 0, st>>>(rowptr, col, order, tile_start, 0, tile, nullptr, ulen, nullptr,
                                                        nullptr, (int32_t *)um.p);
  HIP_TRY(hipGetLastError());
  int32_t umax = 0;
  HIP_TRY(hipMemcpyAsync(&umax, um.p, sizeof(int32_t), hipMemcpyDeviceToHost, st));
  HIP_TRY(hipStreamSynchronize(st));   // the lists may be read on any stream from here on
  if (umax_out) *umax_out = umax;
  if (umax > 65536) INCH_FAIL(INCH_ERR_CAPACITY, "inch_bsr_tiles: a tile's columns span too far or are too many");
  if (ulist && umax > ustride)
    INCH_FAIL(INCH_ERR_CAPACITY, "inch_bsr_tiles: a list of %d columns, room for %d", umax, ustride);
  return INCH_OK;
}

extern "C" inch_status inch_anm_tile_order(int64_t n, const double *xyz, double side, int32_t tile, int32_t *order,
                                           int32_t *tile_start, int64_t *ntile_out, void *stream) {
  INCH_REQUIRE(n > 0 && n < (int64_t)1 << 31 && xyz && order && tile_start && ntile_out && side > 0 && tile > 0,
               "inch_anm_tile_order: bad args");
  hipStream_t st = (hipStream_t)stream;
  const int bs = 256;
  const int nb = 256;
  DevBuf part;
  HIP_TRY(hipMalloc(&part.p, nb * 6 * sizeof(double)));
  k_minmax<<<nb, 256, 0, st>>>(n, xyz, (double *)part.p);
  HIP_TRY(hipGetLastError());
  std::vector<double> hp(nb * 6);
  HIP_TRY(hipMemcpyAsync(hp.data(), part.p, nb * 6 * sizeof(double), hipMemcpyDeviceToHost, st));
  HIP_TRY(hipStreamSynchronize(st));
  CGrid g;
  double hi[3];
  for (int a = 0; a < 3; ++a) {
    g.lo[a] = INFINITY;
    hi[a] = -INFINITY;
    bool nan = false;   // std::min/max would drop a NaN partial
    for (int b = 0; b < nb; ++b) {
      nan |= std::isnan(hp[b * 6 + a]) || std::isnan(hp[b * 6 + 3 + a]);
      g.lo[a] = std::min(g.lo[a], hp[b * 6 + a]);
      hi[a] = std::max(hi[a], hp[b * 6 + 3 + a]);
    }
    if (nan || !std::isfinite(g.lo[a]) || !std::isfinite(hi[a])) INCH_FAIL(INCH_ERR_NAN, "inch_anm_tile_order: non-finite coordinates");
    // an infinite span has no finite number of columns, however wide they are
    if (a < 2 && !std::isfinite(hi[a] - g.lo[a]))
      INCH_FAIL(INCH_ERR_CAPACITY, "inch_anm_tile_order: the coordinates' span overflows");
  }
  // columns (coarser ones where their numbers would not fit 31 bits)
  for (double s = side;; s *= 2.0) {
    double cells = 1.0;
    for (int a = 0; a < 2; ++a) {
      g.inv[a] = 1.0 / s;
      const double d = std::floor((hi[a] - g.lo[a]) * g.inv[a]) + 1.0;
      cells *= d;
      g.dim[a] = d < 2147483647.0 ? std::max<int64_t>(1, (int64_t)d) : (int64_t)1 << 31;
    }
    if (cells < 2147483647.0) break;
  }
  const double zspan = hi[2] - g.lo[2], zscale = zspan > 0.0 ? 4294967295.0 / zspan : 0.0;
  DevBuf key, key2, at, head, cidx, first, tiles, base, tmp;
  HIP_TRY(hipMalloc(&key.p, n * sizeof(uint64_t)));
  HIP_TRY(hipMalloc(&key2.p, n * sizeof(uint64_t)));
  HIP_TRY(hipMalloc(&at.p, n * sizeof(int32_t)));
  HIP_TRY(hipMalloc(&head.p, n * sizeof(int32_t)));
  HIP_TRY(hipMalloc(&cidx.p, (n + 1) * sizeof(int32_t)));
  HIP_TRY(hipMalloc(&first.p, (n + 1) * sizeof(int32_t)));
  HIP_TRY(hipMalloc(&base.p, (n + 1) * sizeof(int32_t)));
  const unsigned gb = (unsigned)((n + bs - 1) / bs);
  k_tile_keys<<<gb, bs, 0, st>>>(n, xyz, g, zscale, (uint64_t *)key.p, (int32_t *)at.p);
  HIP_TRY(hipGetLastError());
  int top = 33;
  while (top < 64 && ((uint64_t)(g.dim[0] * g.dim[1]) >> (top - 32))) ++top;
  size_t tmp_bytes = 0;
  HIP_TRY(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp_bytes, (const uint64_t *)key.p, (uint64_t *)key2.p,
                                             (const int32_t *)at.p, order, (int)n, 0, top, st));
  HIP_TRY(hipMalloc(&tmp.p, tmp_bytes));
  HIP_TRY(hipcub::DeviceRadixSort::SortPairs(tmp.p, tmp_bytes, (const uint64_t *)key.p, (uint64_t *)key2.p,
                                             (const int32_t *)at.p, order, (int)n, 0, top, st));
  k_tile_heads<<<gb, bs, 0, st>>>(n, (const uint64_t *)key2.p, (int32_t *)head.p);
  HIP_TRY(hipGetLastError());
  SCAN_TRY(n, (const int32_t *)head.p, (int32_t *)cidx.p);
  k_tile_first<<<gb, bs, 0, st>>>(n, (const int32_t *)head.p, (const int32_t *)cidx.p, (int32_t *)first.p);
  k_tile_column<<<gb, bs, 0, st>>>(n, tile, (const int32_t *)cidx.p, (const int32_t *)first.p, (int32_t *)head.p);
  HIP_TRY(hipGetLastError());
  SCAN_TRY(n, (const int32_t *)head.p, (int32_t *)base.p);
  k_tile_cut<<<gb, bs, 0, st>>>(n, (const int32_t *)cidx.p, (const int32_t *)first.p, (const int32_t *)base.p, tile_start);
  HIP_TRY(hipGetLastError());
  int32_t nt = 0;
  HIP_TRY(hipMemcpyAsync(&nt, (const int32_t *)base.p + n, sizeof(nt), hipMemcpyDeviceToHost, st));
  HIP_TRY(hipStreamSynchronize(st));
  *ntile_out = nt;
  return INCH_OK;
}

extern "C" inch_status inch_anm_tiles(int64_t n, const double *xyz, const int64_t *rowptr, const int32_t *col,
                                      const uint16_t *images, double box_x, double box_y, int64_t ntile,
                                      int32_t tile, int32_t lanes, const int32_t *order, const int32_t *tile_start,
                                      int32_t *tile_atoms, int32_t *slot_of, int32_t *waves, int64_t *blocks_out,
                                      int32_t ucap, int32_t *ulen, uint32_t *ulist, uint16_t *pairs,
                                      int64_t pair_blocks, double *rec, int32_t *umax_out, void *stream) {
  INCH_REQUIRE(n > 0 && xyz && rowptr && col && tile_atoms && slot_of && waves && ntile > 0, "inch_anm_tiles: bad args");
  INCH_REQUIRE(inch_tile_shape_ok(tile, lanes), "inch_anm_tiles: no tile shape of %d atoms x %d lanes", tile, lanes);
  const int64_t slots = ntile * tile, nw = slots * lanes / 64;
  if (48 * slots > (int64_t)UINT32_MAX)
    INCH_FAIL(INCH_ERR_CAPACITY, "inch_anm_tiles: %lld atoms exceed the 32-bit record offsets", (long long)n);
  hipStream_t st = (hipStream_t)stream;
  const int bs = 256;
  DevBuf flags;
  HIP_TRY(hipMalloc(&flags.p, 2 * sizeof(int32_t)));
  HIP_TRY(hipMemsetAsync(flags.p, 0, 2 * sizeof(int32_t), st));
  int32_t *umax = (int32_t *)flags.p + 1;
  int32_t fl[2] = {0, 0};
  auto check = [&]() -> inch_status {
    HIP_TRY(hipMemcpyAsync(fl, flags.p, sizeof(fl), hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    if (fl[0] & 8) INCH_FAIL(INCH_ERR_INVALID, "inch_anm_tiles: a column lies outside [0, n)");
    if (fl[0] & 16) INCH_FAIL(INCH_ERR_CAPACITY, "inch_anm_tiles: squared distances outside 1e-30 .. 1e30, or x beyond 1e150");
    if (fl[0] & 1) INCH_FAIL(INCH_ERR_CAPACITY, "inch_anm_tiles: a tile's neighbours exceed %d", ucap);
    return INCH_OK;
  };
  if (pairs) {   // second call
    INCH_REQUIRE(ulen && ulist && rec && umax_out && ucap > 0 && ucap <= inch_tile_max_union(tile),
                 "inch_anm_tiles: bad args of the fill call");
    INCH_REQUIRE(blocks_out && *blocks_out <= pair_blocks, "inch_anm_tiles: pairs too small");
    k_tile_coords<<<(unsigned)((slots + bs - 1) / bs), bs, 0, st>>>(slots, tile_atoms, xyz, rec, (int32_t *)flags.p);
    HIP_TRY(hipGetLastError());
    if (images)
      k_tile_fill<true><<<(unsigned)ntile, 256, 0, st>>>(n, tile, lanes, xyz, rowptr, col, images, box_x, box_y,
                                                         tile_atoms, slot_of, (const int2 *)waves, ucap, ulen, ulist,
                                                         pairs, (int32_t *)flags.p, umax);
    else
      k_tile_fill<false><<<(unsigned)ntile, 256, 0, st>>>(n, tile, lanes, xyz, rowptr, col, images, 0.0, 0.0,
                                                          tile_atoms, slot_of, (const int2 *)waves, ucap, ulen, ulist,
                                                          pairs, (int32_t *)flags.p, umax);
    HIP_TRY(hipGetLastError());
    const inch_status s = check();
    if (s != INCH_OK) return s;
    *umax_out = fl[1];
    return INCH_OK;
  }
  INCH_REQUIRE(blocks_out && order && tile_start, "inch_anm_tiles: bad args of the first call");
  DevBuf cnt, passes, blocks, ptr;
  HIP_TRY(hipMalloc(&cnt.p, n * sizeof(int32_t)));
  HIP_TRY(hipMalloc(&passes.p, nw * sizeof(int32_t)));
  HIP_TRY(hipMalloc(&blocks.p, nw * sizeof(int32_t)));
  HIP_TRY(hipMalloc(&ptr.p, (nw + 1) * sizeof(int32_t)));
  const unsigned cg = (unsigned)((16 * n + bs - 1) / bs);
  const int most = inch_tile_max_union(tile);
  if (images)
    k_tile_count<true><<<cg, bs, 0, st>>>(n, xyz, rowptr, col, images, box_x, box_y, most, (int32_t *)cnt.p,
                                          (int32_t *)flags.p);
  else
    k_tile_count<false><<<cg, bs, 0, st>>>(n, xyz, rowptr, col, images, 0.0, 0.0, most, (int32_t *)cnt.p,
                                           (int32_t *)flags.p);
  HIP_TRY(hipGetLastError());
  k_tile_slots<<<(unsigned)ntile, 64, 0, st>>>(tile, lanes, order, tile_start, (const int32_t *)cnt.p, tile_atoms, slot_of,
                                               (int32_t *)passes.p, (int32_t *)blocks.p);
  HIP_TRY(hipGetLastError());
  SCAN_TRY(nw, (const int32_t *)blocks.p, (int32_t *)ptr.p);
  k_tile_waves<<<(unsigned)((nw + bs - 1) / bs), bs, 0, st>>>(nw, (const int32_t *)ptr.p, (const int32_t *)passes.p,
                                                              (int2 *)waves);
  HIP_TRY(hipGetLastError());
  int32_t total = 0;
  HIP_TRY(hipMemcpyAsync(&total, (const int32_t *)ptr.p + nw, sizeof(total), hipMemcpyDeviceToHost, st));
  const inch_status s = check();   // syncs
  if (s != INCH_OK) return s;
  *blocks_out = total;
  return INCH_OK;
}
