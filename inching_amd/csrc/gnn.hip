// Coordinate-graph network kernels (learned warm start): dense layers with float16
// weights/activations and float32 accumulation, neighbour-mean aggregation over the ANM
// neighbour graph, and their backward passes. Deterministic: every reduction over atoms
// is two-phase with fixed orders; no atomics.
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include "common.h"

#define HIP_TRY(expr)                                                                      \
  do {                                                                                     \
    hipError_t _e = (expr);                                                                \
    if (_e != hipSuccess) INCH_FAIL(INCH_ERR_HIP, "%s: %s", #expr, hipGetErrorString(_e)); \
  } while (0)

namespace {

constexpr int kMaxD = 96;        // layer widths handled by the kernels
constexpr int kRows = 32;        // rows of a workgroup's tile
constexpr int kPartBlocks = 256; // most workgroups (partials) of a weight gradient

// 16-bit or float weights, rounded to float16
__device__ __forceinline__ float w_half(const __half *w, int64_t q) { return __half2float(w[q]); }
__device__ __forceinline__ float w_half(const float *w, int64_t q) { return __half2float(__float2half(w[q])); }

// acc[r][c] += sum_k x[row0 + r][k] w[k][4 c0 ..] over a tile in LDS: 2 rows x 4 outputs per thread,
// k ascending, one FMA each.
__device__ __forceinline__ void tile_mac(const float *xs, int xp, const float *ws, int wp, int K, int row, int col,
                                         float (&acc)[2][4]) {
  const float *x0 = xs + row * xp, *x1 = x0 + xp;
  for (int k = 0; k < K; ++k) {
    const float4 w = *(const float4 *)(ws + k * wp + col);
    const float a = x0[k], b = x1[k];
    acc[0][0] = __builtin_fmaf(a, w.x, acc[0][0]);
    acc[0][1] = __builtin_fmaf(a, w.y, acc[0][1]);
    acc[0][2] = __builtin_fmaf(a, w.z, acc[0][2]);
    acc[0][3] = __builtin_fmaf(a, w.w, acc[0][3]);
    acc[1][0] = __builtin_fmaf(b, w.x, acc[1][0]);
    acc[1][1] = __builtin_fmaf(b, w.y, acc[1][1]);
    acc[1][2] = __builtin_fmaf(b, w.z, acc[1][2]);
    acc[1][3] = __builtin_fmaf(b, w.w, acc[1][3]);
  }
}

// Forward of a dense layer (NM = 1) or a graph layer (NM = 2, the second input the neighbour
// mean): pre = (b + X0 W0) + X1 W1, every sum in ascending k as one FMA chain from b (from 0 for
// the second), y = pre or its positive part. A workgroup stages 32 rows and the weights in LDS;
// a thread forms 2 rows x 4 outputs at a time, so that 8 FMAs share one 16-byte and two 4-byte
// LDS reads (one output per thread took two reads each and ran at the LDS rate: 12,007 rows of
// 64 x 64 in 26 us per product; both products, their sum and the activation now take 22).
// W0c, W1c (optional): the weights as used, in float16, written by the first workgroup.
template <int NM, typename W>
__global__ void __launch_bounds__(256) k_layer_fwd(int64_t N, int Din, int Dout, const __half *__restrict__ X0,
                                                   const __half *__restrict__ X1, const W *__restrict__ W0,
                                                   const W *__restrict__ W1, const float *__restrict__ b, int relu,
                                                   float *__restrict__ pre, __half *__restrict__ Y16,
                                                   float *__restrict__ Y32, __half *__restrict__ W0c,
                                                   __half *__restrict__ W1c) {
  extern __shared__ float sm[];
  const int wp = (Dout + 3) & ~3, xp = Din + 1, tid = threadIdx.x;
  float *ws[NM], *xs[NM];
  const __half *X[2] = {X0, X1};
  const W *Wg[2] = {W0, W1};
  __half *Wc[2] = {W0c, W1c};
  const int64_t r0 = (int64_t)blockIdx.x * kRows;
#pragma unroll
  for (int m = 0; m < NM; ++m) {
    ws[m] = sm + m * Din * wp;
    xs[m] = sm + NM * Din * wp + m * kRows * xp;
    for (int t = tid; t < Din * wp; t += 256) {
      const int k = t / wp, o = t - k * wp;
      const float w = o < Dout ? w_half(Wg[m], (int64_t)k * Dout + o) : 0.f;
      ws[m][t] = w;
      if (Wc[m] && blockIdx.x == 0 && o < Dout) Wc[m][k * Dout + o] = __float2half(w);
    }
    for (int t = tid; t < kRows * Din; t += 256) {
      const int r = t / Din, k = t - r * Din;
      xs[m][r * xp + k] = r0 + r < N ? __half2float(X[m][(r0 + r) * Din + k]) : 0.f;
    }
  }
  __syncthreads();
  const int groups = wp / 4;
  for (int t = tid; t < (kRows / 2) * groups; t += 256) {
    const int row = 2 * (t / groups), col = 4 * (t % groups);
    float acc[2][4];
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[0][c] = acc[1][c] = (b && col + c < Dout) ? b[col + c] : 0.f;
    tile_mac(xs[0], xp, ws[0], wp, Din, row, col, acc);
    if constexpr (NM == 2) {
      float ac2[2][4] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
      tile_mac(xs[1], xp, ws[1], wp, Din, row, col, ac2);
#pragma unroll
      for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[r][c] += ac2[r][c];
    }
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      if (r0 + row + r >= N) continue;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        if (col + c >= Dout) continue;
        const int64_t q = (r0 + row + r) * Dout + col + c;
        const float v = (relu && acc[r][c] < 0.f) ? 0.f : acc[r][c];
        if (pre) pre[q] = acc[r][c];
        if (Y16) Y16[q] = __float2half(v);
        if (Y32) Y32[q] = v;
      }
    }
  }
}

// Backward of the same: dP = dY (masked to pre > 0 when pre is given), dX_m = dP W_m^T (o
// ascending, one FMA each), and per workgroup the partial sums of dW_m = X_m^T dP and db = sum dP
// over its tiles of 32 rows: part[block] = [dW_0 | dW_1 | db]; winv (optional): the rows' 1 / (deg - 1). Everything is read once. The
// weight gradient is a 16 x 16 grid of threads with MI x MO outputs each in registers (MI * MO
// FMAs per MI + MO LDS reads), the input gradient 2 rows x 4 inputs per thread against the
// transposed weights. At 12,007 rows of 64 x 64 the separate kernels took 108 us (dX: its LDS
// reads of the weights collided 32 ways) and 82 us (dW: one output per thread, serial over a
// block's rows, from memory) per product; the fused kernel takes 64 us for both.
template <int NM, int MI, int MO>
__global__ void __launch_bounds__(256) k_layer_bwd(int64_t N, int Din, int Dout, const __half *__restrict__ X0,
                                                   const __half *__restrict__ X1, const __half *__restrict__ W0,
                                                   const __half *__restrict__ W1, const float *__restrict__ pre,
                                                   const float *__restrict__ dY, float *__restrict__ dX0,
                                                   float *__restrict__ dX1, float *__restrict__ part,
                                                   const int64_t *__restrict__ rowptr, float *__restrict__ winv) {
  extern __shared__ float sm[];
  const int ip = (Din + 3) & ~3, op = Dout + 1, tid = threadIdx.x;
  float *wt[NM], *xs[NM];
  float *dp = sm;                                   // [kRows][op]
  float *next = sm + ((kRows * op + 3) & ~3);
  const __half *X[2] = {X0, X1};
  const __half *Wg[2] = {W0, W1};
  float *dX[2] = {dX0, dX1};
#pragma unroll
  for (int m = 0; m < NM; ++m) {
    wt[m] = next;                                   // [Dout][ip], transposed
    next += Dout * ip;
    xs[m] = next;                                   // [kRows][ip]
    next += kRows * ip;
    for (int t = tid; t < Dout * ip; t += 256) {
      const int k = t / Dout, o = t - k * Dout;     // consecutive threads read consecutive o
      wt[m][o * ip + k] = k < Din ? __half2float(Wg[m][k * Dout + o]) : 0.f;
    }
  }
  const int tx = tid & 15, ty = tid >> 4;
  float acc[NM][MI][MO];
  float bs = 0.f;
#pragma unroll
  for (int m = 0; m < NM; ++m)
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int o = 0; o < MO; ++o) acc[m][i][o] = 0.f;
  const int64_t ntile = (N + kRows - 1) / kRows;
  for (int64_t tile = blockIdx.x; tile < ntile; tile += gridDim.x) {
    const int64_t r0 = tile * kRows;
    if (winv && tid < kRows && r0 + tid < N) {
      const int64_t d = rowptr[r0 + tid + 1] - rowptr[r0 + tid] - 1;
      winv[r0 + tid] = d > 0 ? 1.f / (float)d : 0.f;
    }
    __syncthreads();
    for (int t = tid; t < kRows * Dout; t += 256) {
      const int r = t / Dout, o = t - r * Dout;
      const int64_t q = (r0 + r) * Dout + o;
      float v = r0 + r < N ? dY[q] : 0.f;
      if (pre && r0 + r < N && !(pre[q] > 0.f)) v = 0.f;
      dp[r * op + o] = v;
    }
#pragma unroll
    for (int m = 0; m < NM; ++m)
      for (int t = tid; t < kRows * Din; t += 256) {
        const int r = t / Din, k = t - r * Din;
        xs[m][r * ip + k] = r0 + r < N ? __half2float(X[m][(r0 + r) * Din + k]) : 0.f;
      }
    __syncthreads();
    const int groups = ip / 4;
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      if (!dX[m]) continue;
      for (int t = tid; t < (kRows / 2) * groups; t += 256) {
        const int row = 2 * (t / groups), col = 4 * (t % groups);
        float a[2][4] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
        tile_mac(dp, op, wt[m], ip, Dout, row, col, a);
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
          for (int c = 0; c < 4; ++c)
            if (r0 + row + r < N && col + c < Din) dX[m][(r0 + row + r) * Din + col + c] = a[r][c];
      }
    }
    for (int r = 0; r < kRows; ++r) {
      float d[MO];
#pragma unroll
      for (int o = 0; o < MO; ++o) d[o] = tx + 16 * o < Dout ? dp[r * op + tx + 16 * o] : 0.f;
#pragma unroll
      for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int i = 0; i < MI; ++i) {
          const float x = ty + 16 * i < Din ? xs[m][r * ip + ty + 16 * i] : 0.f;
#pragma unroll
          for (int o = 0; o < MO; ++o) acc[m][i][o] = __builtin_fmaf(x, d[o], acc[m][i][o]);
        }
    }
    if (tid < Dout)
      for (int r = 0; r < kRows; ++r) bs += dp[r * op + tid];
  }
  float *dst = part + (int64_t)blockIdx.x * (NM * Din * Dout + Dout);
#pragma unroll
  for (int m = 0; m < NM; ++m)
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int o = 0; o < MO; ++o)
        if (ty + 16 * i < Din && tx + 16 * o < Dout)
          dst[m * Din * Dout + (ty + 16 * i) * Dout + tx + 16 * o] = acc[m][i][o];
  if (tid < Dout) dst[NM * Din * Dout + tid] = bs;
}

// Sums of the per-workgroup partials in a fixed order: 32 outputs per workgroup, 8 threads each
// over every 8th partial, their sums added in order (one thread per output waited for 256
// dependent loads: 44 us).
__global__ void __launch_bounds__(256) k_sum_part(int nparts, int m, int n0, int n1, const float *__restrict__ part,
                                                  float *__restrict__ out0, float *__restrict__ out1,
                                                  float *__restrict__ outb) {
  __shared__ float red[8][32];
  const int c = threadIdx.x & 31, g = threadIdx.x >> 5;
  const int j = blockIdx.x * 32 + c;
  float s = 0.f;
  if (j < m) {
#pragma unroll 8
    for (int p = g; p < nparts; p += 8) s += part[(int64_t)p * m + j];
  }
  red[g][c] = s;
  __syncthreads();
  if (g || j >= m) return;
#pragma unroll
  for (int q = 1; q < 8; ++q) s += red[q][c];
  if (j < n0)
    out0[j] = s;
  else if (j < n0 + n1)
    out1[j - n0] = s;
  else
    outb[j - n0 - n1] = s;
}

// mode 0 (forward):  Y[i] = sum_{j in N(i), j != i} X[j] / (deg_i - 1)
// mode 1 (adjoint):  Y[i] = sum_{j in N(i), j != i} X[j] / (deg_j - 1)   (N symmetric)
// add (optional): Y[i] = add[i] + the sum. L lanes per row with V features each; a row's
// neighbours are summed in the list's order, 8 gathers in flight and the next 8 numbers behind
// them (one wave per row and one gather at a time took 60 us at 12,007 rows of 64 float16, now
// 29; the float32 adjoint 102, now 30, with the neighbours' weights from winv when given).
template <typename T, int V>
struct alignas(V * sizeof(T)) Feat {
  T v[V];
};

template <typename T, typename O, int V>
__global__ void __launch_bounds__(256) k_aggregate(int64_t N, int D, int L, const int64_t *__restrict__ rowptr,
                                                   const int32_t *__restrict__ col, const T *__restrict__ X,
                                                   O *__restrict__ Y, int mode, const float *__restrict__ winv,
                                                   const O *__restrict__ add) {
  constexpr int U = 8;
  const int64_t i = (blockIdx.x * (int64_t)256 + threadIdx.x) / L;
  const int l = threadIdx.x % L;
  if (i >= N) return;
  const int64_t b0 = rowptr[i], b1 = rowptr[i + 1];
  const float inv_i = (b1 - b0 > 1) ? 1.f / (float)(b1 - b0 - 1) : 0.f;
  for (int d = V * l; d < D; d += V * L) {
    float acc[V];
#pragma unroll
    for (int c = 0; c < V; ++c) acc[c] = 0.f;
    int32_t jn[U];
#pragma unroll
    for (int q = 0; q < U; ++q) jn[q] = b0 + q < b1 ? col[b0 + q] : (int32_t)i;
    for (int64_t b = b0; b < b1; b += U) {
      int32_t j[U];
      Feat<T, V> x[U];
      float w[U];
#pragma unroll
      for (int q = 0; q < U; ++q) {
        j[q] = jn[q];
        x[q] = *(const Feat<T, V> *)(X + (int64_t)j[q] * D + d);
        if (mode == 1) {
          if (winv) {
            w[q] = winv[j[q]];
          } else {
            const int64_t dj = rowptr[j[q] + 1] - rowptr[j[q]] - 1;
            w[q] = dj > 0 ? 1.f / (float)dj : 0.f;
          }
        }
      }
      // the next neighbours' numbers are in flight with this round's gathers
#pragma unroll
      for (int q = 0; q < U; ++q) jn[q] = b + U + q < b1 ? col[b + U + q] : (int32_t)i;
#pragma unroll
      for (int q = 0; q < U; ++q)
#pragma unroll
        for (int c = 0; c < V; ++c)
          if (j[q] != i) acc[c] = mode == 1 ? __builtin_fmaf(w[q], (float)x[q].v[c], acc[c]) : acc[c] + (float)x[q].v[c];
    }
#pragma unroll
    for (int c = 0; c < V; ++c) {
      if (mode == 0) acc[c] *= inv_i;
      Y[i * D + d + c] = add ? (O)((float)add[i * D + d + c] + acc[c]) : (O)acc[c];
    }
  }
}

// V features per lane need rows of whole V-feature groups and the group's alignment
template <typename T, typename O>
void launch_aggregate(int64_t N, int D, const int64_t *rowptr, const int32_t *col, const T *X, O *Y, int mode,
                      const float *winv, const O *add, hipStream_t st) {
  const bool vec = D % 4 == 0 && (uintptr_t)X % (4 * sizeof(T)) == 0;
  const int need = vec ? D / 4 : D;
  int L = 1;
  while (L < need && L < 64) L <<= 1;
  const unsigned g = (unsigned)((N * L + 255) / 256);
  if (vec)
    k_aggregate<T, O, 4><<<g, 256, 0, st>>>(N, D, L, rowptr, col, X, Y, mode, winv, add);
  else
    k_aggregate<T, O, 1><<<g, 256, 0, st>>>(N, D, L, rowptr, col, X, Y, mode, winv, add);
}

template <int NM, typename W>
inch_status launch_fwd(int64_t N, int Din, int Dout, const __half *X0, const __half *X1, const W *W0, const W *W1,
                       const float *b, int relu, float *pre, __half *Y16, float *Y32, __half *W0c, __half *W1c,
                       hipStream_t st) {
  const size_t lds = sizeof(float) * NM * ((size_t)Din * ((Dout + 3) & ~3) + (size_t)kRows * (Din + 1));
  if (lds > 64 * 1024)
    HIP_TRY(hipFuncSetAttribute((const void *)k_layer_fwd<NM, W>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  k_layer_fwd<NM, W><<<(unsigned)((N + kRows - 1) / kRows), 256, lds, st>>>(N, Din, Dout, X0, X1, W0, W1, b, relu, pre,
                                                                            Y16, Y32, W0c, W1c);
  HIP_TRY(hipGetLastError());
  return INCH_OK;
}

template <int NM>
inch_status launch_bwd(int64_t N, int Din, int Dout, const __half *X0, const __half *X1, const __half *W0,
                       const __half *W1, const float *pre, const float *dY, float *dX0, float *dX1, float *dW0,
                       float *dW1, float *db, float *work, const int64_t *rowptr, float *winv, hipStream_t st) {
  const int ip = (Din + 3) & ~3;
  const size_t lds = sizeof(float) * (((size_t)kRows * (Dout + 1) + 3 & ~(size_t)3) + (size_t)NM * (Dout + kRows) * ip);
  const int64_t tiles = (N + kRows - 1) / kRows;
  const int gx = (int)(tiles < kPartBlocks ? tiles : kPartBlocks);
#define INCH_BWD(MI, MO)                                                                                            \
  do {                                                                                                              \
    if (lds > 64 * 1024)                                                                                            \
      HIP_TRY(hipFuncSetAttribute((const void *)k_layer_bwd<NM, MI, MO>,                                            \
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));                           \
    k_layer_bwd<NM, MI, MO><<<gx, 256, lds, st>>>(N, Din, Dout, X0, X1, W0, W1, pre, dY, dX0, dX1, work, rowptr, winv); \
  } while (0)
  if (Dout <= 64) {
    if (Din <= 16)
      INCH_BWD(1, 4);
    else if (Din <= 64)
      INCH_BWD(4, 4);
    else
      INCH_BWD(6, 4);
  } else {
    if (Din <= 64)
      INCH_BWD(4, 6);
    else
      INCH_BWD(6, 6);
  }
#undef INCH_BWD
  HIP_TRY(hipGetLastError());
  const int nw = Din * Dout, m = NM * nw + Dout;
  k_sum_part<<<(m + 31) / 32, 256, 0, st>>>(gx, m, nw, NM == 2 ? nw : 0, work, dW0, dW1, db);
  HIP_TRY(hipGetLastError());
  return INCH_OK;
}

__global__ void k_relu_bwd(int64_t n, const float *__restrict__ pre, const float *__restrict__ dY,
                           float *__restrict__ dPre) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    dPre[i] = pre[i] > 0.f ? dY[i] : 0.f;
}

}  // namespace

extern "C" {

int64_t inch_gnn_work_size(int32_t Din, int32_t Dout) { return (int64_t)kPartBlocks * (Din * Dout + Dout); }

inch_status inch_gnn_dense_fwd(int64_t N, int32_t Din, int32_t Dout, const void *X, const void *W, const float *b,
                               int32_t relu, float *Ypre, void *Y, float *Y32, void *stream) {
  INCH_REQUIRE(N > 0 && Din > 0 && Dout > 0 && Din <= kMaxD && Dout <= kMaxD && X && W,
               "inch_gnn_dense_fwd: bad args (widths <= 96)");
  return launch_fwd<1, __half>(N, Din, Dout, (const __half *)X, nullptr, (const __half *)W, nullptr, b, relu, Ypre,
                               (__half *)Y, Y32, nullptr, nullptr, (hipStream_t)stream);
}

inch_status inch_gnn_dense_bwd(int64_t N, int32_t Din, int32_t Dout, const void *X, const void *W, const float *dY,
                               float *dX, float *dW, float *db, float *work, void *stream) {
  INCH_REQUIRE(N > 0 && Din > 0 && Dout > 0 && Din <= kMaxD && Dout <= kMaxD && X && W && dY && dW && db && work,
               "inch_gnn_dense_bwd: bad args");
  return launch_bwd<1>(N, Din, Dout, (const __half *)X, nullptr, (const __half *)W, nullptr, nullptr, dY, dX, nullptr,
                       dW, nullptr, db, work, nullptr, nullptr, (hipStream_t)stream);
}

inch_status inch_gnn_layer_fwd(int64_t N, int32_t Din, int32_t Dout, const int64_t *rowptr, const int32_t *col,
                               const void *h, const float *Ws, const float *Wn, const float *b, void *agg, void *Ws16,
                               void *Wn16, float *pre, float *out, void *stream) {
  INCH_REQUIRE(N > 0 && Din > 0 && Dout > 0 && Din <= kMaxD && Dout <= kMaxD && rowptr && col && h && Ws && Wn && b &&
                   agg && agg != h && Ws16 && Wn16 && pre && out,
               "inch_gnn_layer_fwd: bad args (widths <= 96)");
  hipStream_t st = (hipStream_t)stream;
  launch_aggregate<__half, __half>(N, Din, rowptr, col, (const __half *)h, (__half *)agg, 0, nullptr, nullptr, st);
  HIP_TRY(hipGetLastError());
  return launch_fwd<2, float>(N, Din, Dout, (const __half *)h, (const __half *)agg, Ws, Wn, b, 1, pre, nullptr, out,
                              (__half *)Ws16, (__half *)Wn16, st);
}

int64_t inch_gnn_layer_work_size(int64_t N, int32_t Din, int32_t Dout) {
  return (int64_t)kPartBlocks * (2 * Din * Dout + Dout) + (2 * Din + 1) * N;
}

inch_status inch_gnn_layer_bwd(int64_t N, int32_t Din, int32_t Dout, const int64_t *rowptr, const int32_t *col,
                               const void *h, const void *agg, const void *Ws16, const void *Wn16, const float *pre,
                               const float *dout, float *dh, float *dWs, float *dWn, float *db, float *work,
                               void *stream) {
  INCH_REQUIRE(N > 0 && Din > 0 && Dout > 0 && Din <= kMaxD && Dout <= kMaxD && rowptr && col && h && agg && Ws16 &&
                   Wn16 && pre && dout && dWs && dWn && db && work,
               "inch_gnn_layer_bwd: bad args (widths <= 96)");
  hipStream_t st = (hipStream_t)stream;
  float *self = dh ? work + (int64_t)kPartBlocks * (2 * Din * Dout + Dout) : nullptr;
  float *nbr = dh ? self + N * Din : nullptr;
  float *winv = dh ? nbr + N * Din : nullptr;
  const inch_status s =
      launch_bwd<2>(N, Din, Dout, (const __half *)h, (const __half *)agg, (const __half *)Ws16, (const __half *)Wn16,
                    pre, dout, self, nbr, dWs, dWn, db, work, rowptr, winv, st);
  if (s != INCH_OK || !dh) return s;
  launch_aggregate<float, float>(N, Din, rowptr, col, nbr, dh, 1, winv, self, st);
  HIP_TRY(hipGetLastError());
  return INCH_OK;
}

inch_status inch_gnn_aggregate(int64_t N, int32_t D, const int64_t *rowptr, const int32_t *col, const void *X,
                               int32_t xdt, void *Y, int32_t ydt, int32_t mode, void *stream) {
  INCH_REQUIRE(N > 0 && D > 0 && rowptr && col && X && Y && X != Y && (mode == 0 || mode == 1),
               "inch_gnn_aggregate: bad args");
  hipStream_t st = (hipStream_t)stream;
  // dtype codes: 0 float32, 2 float16
  if (xdt == 2 && ydt == 2)
    launch_aggregate<__half, __half>(N, D, rowptr, col, (const __half *)X, (__half *)Y, mode, nullptr, nullptr, st);
  else if (xdt == 0 && ydt == 0)
    launch_aggregate<float, float>(N, D, rowptr, col, (const float *)X, (float *)Y, mode, nullptr, nullptr, st);
  else if (xdt == 2 && ydt == 0)
    launch_aggregate<__half, float>(N, D, rowptr, col, (const __half *)X, (float *)Y, mode, nullptr, nullptr, st);
  else
    INCH_FAIL(INCH_ERR_INVALID, "inch_gnn_aggregate: dtype pair (%d,%d)", xdt, ydt);
  HIP_TRY(hipGetLastError());
  return INCH_OK;
}

inch_status inch_gnn_relu_bwd(int64_t n, const float *pre, const float *dY, float *dPre, void *stream) {
  INCH_REQUIRE(n > 0 && pre && dY && dPre, "inch_gnn_relu_bwd: bad args");
  hipStream_t st = (hipStream_t)stream;
  int64_t g = (n + 255) / 256;
  if (g > 4096) g = 4096;
  k_relu_bwd<<<(unsigned)g, 256, 0, st>>>(n, pre, dY, dPre);
  HIP_TRY(hipGetLastError());
  return INCH_OK;
}

}  // extern "C"
