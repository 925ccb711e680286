// Device parts of the delayed CGS2 step, shared by its whole-vector and its segmented kernels.
// i = J - 1, V[i] is the provisional basis vector, u = Op V[i].
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

namespace dcgs2 {

// Two neighbouring doubles in one load; V, u and the first dof of a range are 8-byte aligned only.
struct __attribute__((packed, aligned(8))) Pair {
  double x, y;
};

__device__ __forceinline__ double block_sum(double v, double *red) {   // 256 threads, red[4]
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

// The workgroups of a grid of 8 ceil(nchunk / 8) x tiles: the row tiles of a chunk follow each other on
// one XCD (workgroups go round the 8 XCDs), so u and w come from its L2 after the first tile.
__device__ __forceinline__ void chunk_and_tile(unsigned tiles, int &c, int &tile) {
  const unsigned k = blockIdx.x >> 3;
  c = (int)(k / tiles * 8 + (blockIdx.x & 7));
  tile = (int)(k % tiles);
}

inline unsigned chunk_tile_grid(int64_t nchunk, int64_t tiles) { return (unsigned)((nchunk + 7) / 8 * 8 * tiles); }

// out[j] = V_j . u and out[J + j] = V_j . w over dofs [b, e) for the rows j0 .. j0 + 7 (256 threads).
__device__ __forceinline__ void dual_dot(int64_t b, int64_t e, int J, int j0, const double *__restrict__ V, int64_t ld,
                                         const double *__restrict__ u, const double *__restrict__ w,
                                         double *__restrict__ out) {
  __shared__ double red[4][16];
  double a[16] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};   // V_j . u, then V_j . w
  // the loads of all rows without a test between them (each would wait for the one before): a tile of fewer
  // than 8 rows takes 1, 2, 4 or 8, the ones past the last repeat it and are dropped
  auto range = [&](auto rows) {
    constexpr int R = decltype(rows)::value;
    const double *row[R];
#pragma unroll
    for (int t = 0; t < R; ++t) row[t] = V + (int64_t)(j0 + t < J ? j0 + t : J - 1) * ld;
    for (int64_t i = b + 2 * (int)threadIdx.x; i < e; i += 512) {
      if (i + 1 < e) {
        const Pair ui = *(const Pair *)(u + i), wi = *(const Pair *)(w + i);
        Pair v[R];
#pragma unroll
        for (int t = 0; t < R; ++t) v[t] = *(const Pair *)(row[t] + i);
#pragma unroll
        for (int t = 0; t < R; ++t) {
          a[t] += v[t].x * ui.x;
          a[t] += v[t].y * ui.y;
          a[8 + t] += v[t].x * wi.x;
          a[8 + t] += v[t].y * wi.y;
        }
      } else {
        const double ui = u[i], wi = w[i];
#pragma unroll
        for (int t = 0; t < R; ++t) {
          const double v = row[t][i];
          a[t] += v * ui;
          a[8 + t] += v * wi;
        }
      }
    }
  };
  const int left = J - j0;
  if (left > 4)
    range(std::integral_constant<int, 8>{});
  else if (left > 2)
    range(std::integral_constant<int, 4>{});
  else if (left > 1)
    range(std::integral_constant<int, 2>{});
  else
    range(std::integral_constant<int, 1>{});
  // 16 sums over the wave: each step gives half of the values to half of the lanes
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int h = 8, m = 32; h > 0; h >>= 1, m >>= 1)
#pragma unroll
    for (int t = 0; t < h; ++t) {
      const double keep = (lane & m) ? a[t + h] : a[t], give = (lane & m) ? a[t] : a[t + h];
      a[t] = keep + __shfl_xor(give, m, 64);
    }
  a[0] += __shfl_xor(a[0], 2, 64);
  a[0] += __shfl_xor(a[0], 1, 64);
  if ((lane & 3) == 0) red[threadIdx.x >> 6][lane >> 2] = a[0];
  __syncthreads();
  const int q = threadIdx.x;
  if (q < 16 && j0 + (q & 7) < J)
    out[(q >> 3) * J + j0 + (q & 7)] = (red[0][q] + red[1][q]) + (red[2][q] + red[3][q]);
}

// Sums of the partials part[c * 2J + .] over chunks c0 .. c1-1 (thread groups over every ngrp-th chunk, then in
// order over the groups), then with (s_0..s_i, g_0..g_{i-1}, -) these sums and v_i = ~v_i - sum g_l V_l:
// coef[i] = v_i . u = s_i - g . s, coef[j] = s_j - coef[i] g_j (j < i), coef[J + l] = g_l and
// *alpha_i = coef[i] - beta_prev g_{i-1} (the one operator term left in a Krylov basis). 1,024 threads, J <= 256.
__device__ __forceinline__ void coefficients(int J, int64_t c0, int64_t c1, const double *__restrict__ part,
                                             const double *__restrict__ beta_prev, double *__restrict__ coef,
                                             double *__restrict__ alpha_i) {
  __shared__ double red[1024];
  const int tid = threadIdx.x, i = J - 1;
  const int width = (2 * J + 63) & ~63, ngrp = 1024 / width;   // width <= 512
  const int o = tid % width, grp = tid / width;
  double sum = 0.0;
  if (o < 2 * J && grp < ngrp) {
#pragma unroll 8
    for (int64_t c = c0 + grp; c < c1; c += ngrp) sum += part[c * 2 * J + o];
  }
  red[tid] = sum;
  __syncthreads();
  if (tid < width)
    for (int q = 1; q < ngrp; ++q) sum += red[q * width + tid];
  __syncthreads();
  if (tid < width) red[tid] = sum;
  __syncthreads();
  if (tid >= 64) return;
  const int lane = tid;
  const double *sv = red, *g = red + J;
  double p = 0.0;
  for (int l = lane; l < i; l += 64) p += g[l] * sv[l];
  for (int off = 32; off > 0; off >>= 1) p += __shfl_xor(p, off, 64);
  const double ci = sv[i] - p;
  for (int j = lane; j < i; j += 64) {
    coef[j] = sv[j] - ci * g[j];
    coef[J + j] = g[j];
  }
  if (lane == 0) {
    coef[i] = ci;
    *alpha_i = i > 0 ? ci - beta_prev[0] * g[i - 1] : ci;
  }
}

// u -= sum_{j<=i} ca[j] V_j and V[i] -= sum_{l<i} cg[l] V_l over dofs [x0, x1) in one read of V[0..i]; returns
// the thread's part of |u'|^2. 256 threads; a thread takes 4 dofs at a time (two pairs), the loads of 4 rows in
// flight; ca and cg are wave-uniform and come by scalar loads.
__device__ __forceinline__ double update(int64_t x0, int64_t x1, int J, double *__restrict__ V, int64_t ld,
                                         const double *__restrict__ ca, const double *__restrict__ cg,
                                         double *__restrict__ u) {
  const int i = J - 1;
  double ss = 0.0;
  int64_t xb = x0;
  for (; xb + 1024 <= x1; xb += 1024) {
    const int64_t x = xb + 2 * (int)threadIdx.x;
    double su[4] = {0, 0, 0, 0}, sv[4] = {0, 0, 0, 0};
    const double *Vx = V + x;
#pragma unroll 4
    for (int j = 0; j < i; ++j) {
      const Pair v0 = *(const Pair *)(Vx + (int64_t)j * ld), v1 = *(const Pair *)(Vx + (int64_t)j * ld + 512);
      const double a = ca[j], g = cg[j];
      su[0] += a * v0.x, su[1] += a * v0.y, su[2] += a * v1.x, su[3] += a * v1.y;
      sv[0] += g * v0.x, sv[1] += g * v0.y, sv[2] += g * v1.x, sv[3] += g * v1.y;
    }
    const double ai = ca[i];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      Pair *vp = (Pair *)(V + (int64_t)i * ld + x + 512 * h), *up = (Pair *)(u + x + 512 * h);
      const Pair vi = *vp, uo = *up;
      const Pair un = {uo.x - (su[2 * h] + ai * vi.x), uo.y - (su[2 * h + 1] + ai * vi.y)};
      *up = un;
      *vp = {vi.x - sv[2 * h], vi.y - sv[2 * h + 1]};
      ss += un.x * un.x;
      ss += un.y * un.y;
    }
  }
  for (int64_t x = xb + threadIdx.x; x < x1; x += 256) {   // fewer than 1,024 left
    double su = 0.0, sv = 0.0;
#pragma unroll 8
    for (int j = 0; j < i; ++j) {
      const double v = V[(int64_t)j * ld + x];
      su += ca[j] * v;
      sv += cg[j] * v;
    }
    const double vi = V[(int64_t)i * ld + x];
    const double un = u[x] - (su + ca[i] * vi);
    u[x] = un;
    V[(int64_t)i * ld + x] = vi - sv;
    ss += un * un;
  }
  return ss;
}

// The same over dofs [x, x + 64) cut at x1: one dof per lane, the rows dealt to the four waves (short vectors:
// more workgroups, and a quarter of the rows in each lane's chain).
__device__ __forceinline__ double update_narrow(int64_t x, int64_t x1, int J, double *__restrict__ V, int64_t ld,
                                                const double *__restrict__ ca, const double *__restrict__ cg,
                                                double *__restrict__ u) {
  __shared__ double sums[2][4][64];
  const int i = J - 1, lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  x += lane;
  double su = 0.0, sv = 0.0, vi = 0.0, uo = 0.0;
  if (x < x1) {
    if (w == 0) {
      vi = V[(int64_t)i * ld + x];
      uo = u[x];
    }
#pragma unroll 8
    for (int j = w; j < i; j += 4) {
      const double v = V[(int64_t)j * ld + x];
      su += ca[j] * v;
      sv += cg[j] * v;
    }
  }
  __syncthreads();
  sums[0][w][lane] = su;
  sums[1][w][lane] = sv;
  __syncthreads();
  if (w || x >= x1) return 0.0;
  su = (sums[0][0][lane] + sums[0][1][lane]) + (sums[0][2][lane] + sums[0][3][lane]);
  sv = (sums[1][0][lane] + sums[1][1][lane]) + (sums[1][2][lane] + sums[1][3][lane]);
  const double un = uo - (su + ca[i] * vi);
  u[x] = un;
  V[(int64_t)i * ld + x] = vi - sv;
  return un * un;
}

}  // namespace dcgs2
