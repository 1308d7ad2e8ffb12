// RMSNorm over the last dimension for gfx950: the LM's pre-norms (models/common.py:8-16,
// used at models/lm.py:63,95 and applied at :83,128).
//   y = (x r) w,  r = 1 / sqrt(mean_j x_j^2 + eps)  per row.
// Backward (g = dy w, xhat = x r):
//   dx = r (g - xhat mean_j(g xhat)),   dw = sum over rows of dy xhat.
// NP lanes own a row: lane l holds columns (k NP + l) V + i, i < V, so a wavefront reads 64 / NP
// whole rows in K vector loads per lane, and the row sums are reductions over NP lanes whose result
// every one of them holds bit for bit.  A lane issues the loads of P rows before any arithmetic.
// The backward is persistent: at most kNormBlocks workgroups stride over the rows, keep dw in
// registers and leave one partial row each, which a second kernel adds in workgroup order, in
// float64: no float atomics, bitwise reproducible.
// HBM bounds both directions from some 8 MB on.  Forward, backward, sum of dw in us, from one
// wavefront per row, one column per load and one partial row per 8 to 32 rows:
//   8192 x 256      5.4 +   7.4 +  3.1 ->  5.4 +   6.2 + 2.4   (16.8 and 25.2 MB)
//   8192 x 1024    13.4 +  16.9 +  6.7 -> 12.0 +  17.2 + 3.9   (67 and 101 MB)
//   65536 x 64     13.7 +  10.6 + 10.1 ->  8.1 +  10.5 + 3.9   (a row fills 16 lanes, not 64)
//   65536 x 1024   97.9 + 156.3 + 71.7 -> 87.0 + 152.1 + 4.8   (512 partial rows, not 8192)
#include "ssm_device.hpp"
#include "ssm_internal.hpp"
#include "ssm_tiles.hpp"
#include "ssm_wave.hpp"

namespace ssm {

template <typename T, int V>
__device__ __forceinline__ void cols_load(const T *src, T (&v)[V]) {
  struct alignas(V * sizeof(T)) Pack { T e[V]; };
  const Pack k = *(const Pack *)src;
#pragma unroll
  for (int i = 0; i < V; ++i) v[i] = k.e[i];
}
template <typename T, int V>
__device__ __forceinline__ void cols_store(T *dst, const T (&v)[V]) {
  struct alignas(V * sizeof(T)) Pack { T e[V]; };
  Pack k;
#pragma unroll
  for (int i = 0; i < V; ++i) k.e[i] = v[i];
  *(Pack *)dst = k;
}
// The lane's columns of one row (0 past the end).
template <typename T, int V, int NP, int K>
__device__ __forceinline__ void row_cols(const T *row, int l, int C, T (&v)[K][V]) {
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int j = (k * NP + l) * V;
    if (j < C) {
      cols_load<T, V>(row + j, v[k]);
    } else {
#pragma unroll
      for (int i = 0; i < V; ++i) v[k][i] = 0;
    }
  }
}

template <typename T, int V, int NP, int K, int P>
__global__ void __launch_bounds__(kNormThreads) k_norm_fwd(const NormParams p) {
  constexpr int RL = kNormThreads / NP;  // rows of one pass
  const int l = threadIdx.x % NP, C = (int)p.C;
  const int64_t r0 = (int64_t)blockIdx.x * RL * P + threadIdx.x / NP;
  T v[P][K][V], w[K][V];
#pragma unroll
  for (int q = 0; q < P; ++q) {  // rows past the end read the last row and are not used
    const int64_t row = r0 + q * RL < p.R ? r0 + q * RL : p.R - 1;
    row_cols<T, V, NP, K>((const T *)p.x + row * p.sx, l, C, v[q]);
  }
  row_cols<T, V, NP, K>((const T *)p.w, l, C, w);
#pragma unroll
  for (int q = 0; q < P; ++q) {
    const int64_t row = r0 + q * RL;
    T ss = 0;
#pragma unroll
    for (int k = 0; k < K; ++k)
#pragma unroll
      for (int i = 0; i < V; ++i) ss = fma(v[q][k][i], v[q][k][i], ss);
    ss = group_sum<NP>(ss);
    const T r = (T)1 / sqrt(ss / (T)C + (T)p.eps);
    if (row >= p.R) continue;
    if (l == 0) ((T *)p.rstd)[row] = r;
    T *yr = (T *)p.y + row * p.sy;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int j = (k * NP + l) * V;
      T o[V];
#pragma unroll
      for (int i = 0; i < V; ++i) o[i] = (v[q][k][i] * r) * w[k][i];  // the reference's order: (x r), then * w
      if (j < C) cols_store<T, V>(yr + j, o);
    }
  }
}

template <typename T, int V, int NP, int K, int P>
__global__ void __launch_bounds__(kNormBwdThreads) k_norm_bwd(const NormParams p) {
  constexpr int RL = kNormBwdThreads / NP, CP = K * NP * V;  // rows of one pass, columns padded
  __shared__ __align__(16) T red[RL][CP];
  const int l = threadIdx.x % NP, rl = threadIdx.x / NP, C = (int)p.C;
  T w[K][V], acc[K][V];
  row_cols<T, V, NP, K>((const T *)p.w, l, C, w);
#pragma unroll
  for (int k = 0; k < K; ++k)
#pragma unroll
    for (int i = 0; i < V; ++i) acc[k][i] = 0;
  for (int64_t base = (int64_t)blockIdx.x * RL * P; base < p.R; base += (int64_t)gridDim.x * RL * P) {
    T xv[P][K][V], dv[P][K][V], rs[P];
#pragma unroll
    for (int q = 0; q < P; ++q) {  // rows past the end read the last row and are not used
      const int64_t row = base + q * RL + rl < p.R ? base + q * RL + rl : p.R - 1;
      rs[q] = ((const T *)p.rstd)[row];
      row_cols<T, V, NP, K>((const T *)p.x + row * p.sx, l, C, xv[q]);
      row_cols<T, V, NP, K>((const T *)p.dy + row * p.sdy, l, C, dv[q]);
    }
#pragma unroll
    for (int q = 0; q < P; ++q) {
      const int64_t row = base + q * RL + rl;
      const T r = rs[q];
      T dot = 0;
#pragma unroll
      for (int k = 0; k < K; ++k)
#pragma unroll
        for (int i = 0; i < V; ++i) dot = fma(dv[q][k][i] * w[k][i], xv[q][k][i] * r, dot);
      const T c = group_sum<NP>(dot) / (T)C;
      if (row >= p.R) continue;
      T *dxr = (T *)p.dx + row * p.sdx;
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const int j = (k * NP + l) * V;
        T o[V];
#pragma unroll
        for (int i = 0; i < V; ++i) {
          const T xh = xv[q][k][i] * r;
          o[i] = r * (dv[q][k][i] * w[k][i] - xh * c);
          acc[k][i] = fma(dv[q][k][i], xh, acc[k][i]);
        }
        if (j < C) cols_store<T, V>(dxr + j, o);
      }
    }
  }
#pragma unroll
  for (int k = 0; k < K; ++k) cols_store<T, V>(&red[rl][(k * NP + l) * V], acc[k]);
  __syncthreads();
  for (int j = threadIdx.x; j < C; j += kNormBwdThreads) {
    double s = 0;  // up to 64 rows' sums: float32 adds would show in dw
#pragma unroll
    for (int q = 0; q < RL; ++q) s += (double)red[q][j];
    ((T *)p.ws)[(int64_t)blockIdx.x * C + j] = (T)s;
  }
}

// dw_j = sum over the backward's workgroups (in order) of their partials: a workgroup of
// kNormFinThreads lanes per 64 columns, kNormFinThreads / 64 lanes per column each summing a
// contiguous range of partials (16 loads in flight), then those ranges in order.
template <typename T>
__global__ void __launch_bounds__(kNormFinThreads) k_norm_fin(const NormParams p) {
  constexpr int Q = kNormFinThreads / kWave;
  __shared__ double part[Q][kWave];
  const int lane = threadIdx.x % kWave, q = threadIdx.x / kWave;
  const int64_t j = (int64_t)blockIdx.x * kWave + lane;
  const int64_t per = (p.nblk + Q - 1) / Q;
  const int64_t b0 = q * per, b1 = b0 + per < p.nblk ? b0 + per : p.nblk;
  double s = 0;
  if (j < p.C && b0 < b1) s = ordered_sum<16, T, double>((const T *)p.ws + b0 * p.C + j, p.C, b1 - b0);
  part[q][lane] = s;
  __syncthreads();
  if (q == 0 && j < p.C) {
    double t = 0;
#pragma unroll
    for (int k = 0; k < Q; ++k) t += part[k][lane];
    ((T *)p.dw)[j] = (T)t;
  }
}

template <typename T, int V, int NP, int K, int P>
static hipError_t norm_v(NormParams p, bool bwd, hipStream_t s) {
  constexpr int64_t fr = kNormThreads / NP * P, br = kNormBwdThreads / NP * P;  // rows per workgroup and pass
  if (!bwd) {
    hipLaunchKernelGGL((k_norm_fwd<T, V, NP, K, P>), dim3((unsigned)((p.R + fr - 1) / fr)), dim3(kNormThreads), 0, s, p);
    return hipGetLastError();
  }
  static_assert(br >= norm_bwd_rows(K * NP * V), "the partials' workspace");
  p.nblk = (p.R + br - 1) / br < kNormBlocks ? (p.R + br - 1) / br : kNormBlocks;
  hipLaunchKernelGGL((k_norm_bwd<T, V, NP, K, P>), dim3((unsigned)p.nblk), dim3(kNormBwdThreads), 0, s, p);
  hipLaunchKernelGGL((k_norm_fin<T>), dim3((unsigned)((p.C + kWave - 1) / kWave)), dim3(kNormFinThreads), 0, s, p);
  return hipGetLastError();
}

// Any C and alignment: one column per load, a wavefront per row.  Forward + backward + sum in us,
// unaligned rows, from one partial row per 8 to 32 rows: 8192 x 201 5.1 + 7.6 + 3.1 -> 5.2 + 6.1 + 2.6,
// 8192 x 1001 13.1 + 17.2 + 6.8 -> 11.3 + 17.3 + 3.8, 65536 x 63 13.8 + 11.5 + 11.6 -> 10.9 + 12.4 + 3.7;
// float64 8192 x 512 12.4 + 18.1 + 5.0 -> 12.4 + 19.6 + 5.2, 65536 x 1024 188 + 302 + 94 -> 181 + 313 + 7.
template <typename T>
static hipError_t norm_c1(const NormParams &p, bool bwd, hipStream_t s) {
  if (p.C <= 64) return norm_v<T, 1, 64, 1, 4>(p, bwd, s);
  if (p.C <= 128) return norm_v<T, 1, 64, 2, 4>(p, bwd, s);
  if (p.C <= 256) return norm_v<T, 1, 64, 4, 4>(p, bwd, s);
  if (p.C <= 512) return norm_v<T, 1, 64, 8, 2>(p, bwd, s);
  return p.C <= kNormMaxC ? norm_v<T, 1, 64, 16, 1>(p, bwd, s) : hipErrorInvalidValue;
}

// float32 rows of whole, 16-byte aligned groups of four columns: the fewest lanes that hold a row in
// one load each (so that short rows fill the wavefront too), 16 columns of loads in flight per lane.
// Against one column per load, forward: 8192 x 200 4.7 -> 4.9 us, 8192 x 512 9.0 -> 7.7, 65536 x 64
// 13.7 -> 8.1, 65536 x 256 23.9 -> 20.7.
static hipError_t norm_c4(const NormParams &p, bool bwd, hipStream_t s) {
  if (p.C <= 32) return norm_v<float, 4, 8, 1, 4>(p, bwd, s);
  if (p.C <= 64) return norm_v<float, 4, 16, 1, 4>(p, bwd, s);
  if (p.C <= 128) return norm_v<float, 4, 32, 1, 4>(p, bwd, s);
  if (p.C <= 256) return norm_v<float, 4, 64, 1, 4>(p, bwd, s);
  if (p.C <= 512) return norm_v<float, 4, 64, 2, 2>(p, bwd, s);
  return p.C <= kNormMaxC ? norm_v<float, 4, 64, 4, 1>(p, bwd, s) : hipErrorInvalidValue;
}

static bool quads(const NormParams &p, const void *ptr, int64_t stride) {
  return (uintptr_t)ptr % 16 == 0 && (p.R == 1 || stride % 4 == 0);
}

hipError_t launch_norm(const NormParams &p, int dtype, bool bwd, hipStream_t s) {
  if (dtype == 3) return norm_c1<double>(p, bwd, s);
  const bool q4 = p.C % 4 == 0 && quads(p, p.w, 0) && quads(p, p.x, p.sx) &&
                  (bwd ? quads(p, p.dy, p.sdy) && quads(p, p.dx, p.sdx) : quads(p, p.y, p.sy));
  return q4 ? norm_c4(p, bwd, s) : norm_c1<float>(p, bwd, s);
}

}  // namespace ssm
