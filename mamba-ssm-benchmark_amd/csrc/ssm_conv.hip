// Causal depthwise conv1d (+ SiLU) for gfx950: the producer of the scan's input in the Mamba
// block, models/mamba.py:101-107:
//   xc = pad_left(x, W-1) (or [state, x]);  out = silu(conv1d(xc, w, bias, groups=D));
//   state <- the last W-1 columns of xc.
// x and out are (B, L, D) views (the in_proj split of models/mamba.py:100 is D-contiguous).
// A workgroup is 64 lanes along D (one channel each: neighbouring lanes make every read coalesced)
// x kConvTG time blocks of kConvTT steps, one wavefront each; a lane reads the W-1 inputs before
// its steps as well (the overlap between time blocks is served from cache).  The kernels are bound
// by HBM once enough wavefronts run; before that, by the instructions of a wavefront's 25 reads:
// the time block is uniform over the wavefront, so row addresses and bounds on time are scalar
// work, interior blocks take no bound at all, and all reads are issued before any arithmetic.
// Because kConvTT >= W-1, only the first time block reads the carried state, and it also writes
// the new state (after reading), so the update can be in place.  The backward recomputes the
// pre-activation for the SiLU derivative, forms dx with the transposed taps, and reduces dweight /
// dbias over the workgroup's time blocks in LDS before writing one partial row per workgroup; a
// second kernel adds the rows in a fixed order.
//
// Forward, backward, sum of the partials in us, W 4, with each lane bounding and addressing its
// own rows -> with the scalar rows:
//   1 x 512 x 512 float32     4.5 +  6.2 +   2.8 ->  3.5 +  4.5 +  2.8
//   16 x 512 x 512 float32   10.0 + 13.8 +   6.3 ->  8.5 + 11.0 to 12.4 + 4.2   (33.6 and 50.3 MB)
//   8 x 1024 x 4096 bf16     62.1 + 119  +   6.9 -> 33.0 + 60.2 +  6.2   (134 and 201 MB)
//   32 x 16384 x 64 float32  46.1 + 81.2 + 334.9 -> 43.1 + 74.7 + 35.0
// Two channels x 16 steps per lane is slower up to 4 M elements (16 x 512 x 512: 11.4 + 15.5) and
// gains only in the backward at 33 M (89 -> 78, bf16 60 -> 52).
#include "ssm_device.hpp"
#include "ssm_internal.hpp"
#include "ssm_tiles.hpp"
#include "ssm_wave.hpp"

namespace ssm {

template <typename CT>
__device__ __forceinline__ CT silu_ct(CT v) {
  return v * sigmoid_ct<CT>(v);
}

constexpr int kConvThreads = kWave * kConvTG;

// Rows s0 .. s0 + NX - 1 of a (B, L, D) view at batch row b, element off of each; zero outside
// 0 .. L-1.  s0 is uniform over the wavefront.  Rows outside are read at a clamped address and dropped.
template <typename IT, int NX>
__device__ __forceinline__ void rows_load(const KView &v, int64_t b, int64_t off, int s0, int L,
                                          typename Conv<IT>::CT (&x)[NX]) {
  const IT *base = vp<IT>(v) + b * v.s0;
  if (s0 >= 0 && s0 + NX <= L) {
#pragma unroll
    for (int k = 0; k < NX; ++k) x[k] = Conv<IT>::load(base + (int64_t)(s0 + k) * v.s1 + off);
    return;
  }
#pragma unroll
  for (int k = 0; k < NX; ++k) {
    const int s = s0 + k, c = s < 0 ? 0 : s < L ? s : L - 1;
    x[k] = Conv<IT>::load(base + (int64_t)c * v.s1 + off);
  }
#pragma unroll
  for (int k = 0; k < NX; ++k)
    if (s0 + k < 0 || s0 + k >= L) x[k] = 0;
}

// input at time s < L of [state, x] for channel d of batch row b
template <typename IT, int W>
__device__ __forceinline__ typename Conv<IT>::CT conv_in(const ConvParams &p, int64_t b, int64_t d, int s) {
  typedef typename Conv<IT>::CT CT;
  if (s >= 0) return Conv<IT>::load(vp<IT>(p.x) + b * p.x.s0 + (int64_t)s * p.x.s1 + d * p.x.s2);
  if (!p.has_sin) return (CT)0;
  return Conv<IT>::load(vp<IT>(p.sin) + b * p.sin.s0 + d * p.sin.s1 + (int64_t)(W - 1 + s) * p.sin.s2);
}

template <typename CT, int W>
__device__ __forceinline__ void taps_load(const ConvParams &p, int64_t d, CT (&w)[W], CT &bias) {
#pragma unroll
  for (int j = 0; j < W; ++j) w[j] = vload<CT>(p.w, d * p.w.s0 + j * p.w.s1);
  bias = p.has_bias ? vload<CT>(p.bias, d * p.bias.s0) : (CT)0;
}

template <typename IT, int W>
__global__ void __launch_bounds__(kConvThreads) k_conv_fwd(const ConvParams p) {
  typedef typename Conv<IT>::CT CT;
  constexpr int TT = kConvTT, NX = TT + W - 1;
  const int lane = threadIdx.x % kWave, tg = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int64_t d = (int64_t)blockIdx.x * kWave + lane;
  const int t0 = ((int)blockIdx.y * kConvTG + tg) * TT;
  const int64_t b = blockIdx.z;
  const int L = (int)p.L;
  if (d >= p.D || t0 >= L) return;
  CT w[W], bias, xin[NX];  // xin[k]: input at time t0 - (W-1) + k
  rows_load<IT, NX>(p.x, b, d * p.x.s2, t0 - (W - 1), L, xin);
  taps_load<CT, W>(p, d, w, bias);
  if constexpr (W > 1) {
    if (p.has_sin && t0 == 0) {
#pragma unroll
      for (int k = 0; k < W - 1; ++k) xin[k] = conv_in<IT, W>(p, b, d, k - (W - 1));
    }
    if (p.has_sout && t0 == 0) {
      // the new state: inputs L-(W-1) .. L-1 of [state, x]; this lane is the only reader of the
      // old state, and it reads before it writes
      CT ns[W - 1];
#pragma unroll
      for (int j = 0; j < W - 1; ++j) ns[j] = conv_in<IT, W>(p, b, d, L - (W - 1) + j);
#pragma unroll
      for (int j = 0; j < W - 1; ++j)
        Conv<IT>::store(vpw<IT>(p.sout) + b * p.sout.s0 + d * p.sout.s1 + j * p.sout.s2, ns[j]);
    }
  }
  IT *ob = vpw<IT>(p.out) + b * p.out.s0;
  const int64_t oo = d * p.out.s2;
#pragma unroll
  for (int tt = 0; tt < TT; ++tt) {
    CT acc = bias;
#pragma unroll
    for (int j = 0; j < W; ++j) acc = fma(w[j], xin[tt + j], acc);
    if (t0 + tt < L) Conv<IT>::store(ob + (int64_t)(t0 + tt) * p.out.s1 + oo, p.silu ? silu_ct(acc) : acc);
  }
}

template <typename IT, int W>
__global__ void __launch_bounds__(kConvThreads) k_conv_bwd(const ConvParams p) {
  typedef typename Conv<IT>::CT CT;
  constexpr int TT = kConvTT, NG = TT + W - 1, NX = TT + 2 * (W - 1);
  __shared__ CT red[kConvTG][W + 1][kWave];
  const int lane = threadIdx.x % kWave, tg = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int64_t d = (int64_t)blockIdx.x * kWave + lane;
  const int t0 = ((int)blockIdx.y * kConvTG + tg) * TT;
  const int64_t b = blockIdx.z;
  const int L = (int)p.L;
  CT dwp[W + 1];  // dweight taps, then dbias
#pragma unroll
  for (int j = 0; j <= W; ++j) dwp[j] = 0;
  if (d < p.D && t0 < L) {
    CT w[W], bias, xin[NX], g[NG];  // xin[k]: input at t0 - (W-1) + k; g[k]: dout x silu' at t0 + k
    rows_load<IT, NX>(p.x, b, d * p.x.s2, t0 - (W - 1), L, xin);
    rows_load<IT, NG>(p.dout, b, d * p.dout.s2, t0, L, g);
    taps_load<CT, W>(p, d, w, bias);
    if constexpr (W > 1) {
      if (p.has_sin && t0 == 0) {
#pragma unroll
        for (int k = 0; k < W - 1; ++k) xin[k] = conv_in<IT, W>(p, b, d, k - (W - 1));
      }
    }
    if (p.silu) {
#pragma unroll
      for (int k = 0; k < NG; ++k) {
        CT pre = bias;
#pragma unroll
        for (int j = 0; j < W; ++j) pre = fma(w[j], xin[k + j], pre);
        const CT sg = sigmoid_ct<CT>(pre);
        g[k] *= sg * ((CT)1 + pre * ((CT)1 - sg));
      }
    }
    IT *dxb = vpw<IT>(p.dx) + b * p.dx.s0;
    const int64_t dxo = d * p.dx.s2;
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) {
      if (t0 + tt >= L) break;  // uniform over the wavefront
      // dx[t] = sum_j w[j] g[t + W-1 - j]
      CT acc = 0;
#pragma unroll
      for (int j = 0; j < W; ++j) acc = fma(w[j], g[tt + W - 1 - j], acc);
      Conv<IT>::store(dxb + (int64_t)(t0 + tt) * p.dx.s1 + dxo, acc);
#pragma unroll
      for (int j = 0; j < W; ++j) dwp[j] = fma(g[tt], xin[tt + j], dwp[j]);
      dwp[W] += g[tt];
    }
  }
#pragma unroll
  for (int j = 0; j <= W; ++j) red[tg][j][lane] = dwp[j];
  __syncthreads();
  // one partial row (W + 1, D) per workgroup: the time blocks in order
  CT *ws = (CT *)p.ws + (b * p.nblk + blockIdx.y) * (W + 1) * p.D;
  for (int e = threadIdx.x; e < (W + 1) * kWave; e += kConvThreads) {
    const int j = e / kWave, l = e % kWave;
    const int64_t dd = (int64_t)blockIdx.x * kWave + l;
    if (dd >= p.D) continue;
    CT sum = 0;
#pragma unroll
    for (int q = 0; q < kConvTG; ++q) sum += red[q][j][l];
    ws[j * p.D + dd] = sum;
  }
}

// dweight / dbias: the B * nblk partial rows summed in a fixed order and in float64.  A workgroup
// owns CW of the (W + 1) D columns; its row groups sum rows g, g + G, ... (16 independent loads in
// flight each), and the groups are added in order.  A chain of reads bounds it, so the columns, not
// the channels, are spread over workgroups, and long sums over more row groups.
constexpr int kConvFinThreads = 1024;

template <typename CT, int CW>
__global__ void __launch_bounds__(kConvFinThreads) k_conv_fin(const ConvParams p) {
  constexpr int G = kConvFinThreads / CW;
  __shared__ double red[G][CW];
  const int l = threadIdx.x, g = threadIdx.y;
  const int64_t cols = (p.W + 1) * p.D, e = (int64_t)blockIdx.x * CW + l, rows = p.B * p.nblk;
  double s = 0;
  if (e < cols && g < rows)
    s = ordered_sum<16, CT, double>((const CT *)p.ws + g * cols + e, G * cols, (rows - g + G - 1) / G);
  red[g][l] = s;
  __syncthreads();
  if (g != 0 || e >= cols) return;
  s = 0;
#pragma unroll 16
  for (int q = 0; q < G; ++q) s += red[q][l];
  const int64_t j = e / p.D, d = e % p.D;
  if (j < p.W) vstore<CT>(p.dw, d * p.dw.s0 + j * p.dw.s1, (CT)s);
  else if (p.has_dbias) vstore<CT>(p.dbias, d * p.dbias.s0, (CT)s);
}

template <typename CT, int CW>
static void conv_fin(const ConvParams &p, hipStream_t s) {
  const int64_t cols = (p.W + 1) * p.D;
  // (CW, row groups) threads: a grid row of 2^32 and more would wrap
  hipLaunchKernelGGL((k_conv_fin<CT, CW>), dim3((unsigned)((cols + CW - 1) / CW)), dim3(CW, kConvFinThreads / CW), 0, s, p);
}

template <typename IT, int W>
static hipError_t conv_t(const ConvParams &p, bool bwd, hipStream_t s) {
  typedef typename Conv<IT>::CT CT;
  static_assert(kConvTT >= W - 1, "one time block holds the carried state");
  const dim3 grid((unsigned)((p.D + kWave - 1) / kWave), (unsigned)p.nblk, (unsigned)p.B);
  if (!bwd) {
    hipLaunchKernelGGL((k_conv_fwd<IT, W>), grid, dim3(kConvThreads), 0, s, p);
  } else {
    hipLaunchKernelGGL((k_conv_bwd<IT, W>), grid, dim3(kConvThreads), 0, s, p);
    // 16 columns x 64 row groups from 1024 rows on (8192 rows x 320 columns: 67 -> 35 us); below,
    // 64 x 16 reads whole 256-byte segments (256 rows x 2560 columns: 4.2 us)
    if (p.B * p.nblk >= 1024) conv_fin<CT, 16>(p, s);
    else conv_fin<CT, 64>(p, s);
  }
  return hipGetLastError();
}

template <typename IT>
static hipError_t conv_w(const ConvParams &p, bool bwd, hipStream_t s) {
  switch (p.W) {
    case 1: return conv_t<IT, 1>(p, bwd, s);
    case 2: return conv_t<IT, 2>(p, bwd, s);
    case 3: return conv_t<IT, 3>(p, bwd, s);
    case 4: return conv_t<IT, 4>(p, bwd, s);
    case 5: return conv_t<IT, 5>(p, bwd, s);
    case 6: return conv_t<IT, 6>(p, bwd, s);
    case 7: return conv_t<IT, 7>(p, bwd, s);
    default: return conv_t<IT, 8>(p, bwd, s);
  }
}

hipError_t launch_conv(const ConvParams &p, int dtype, bool bwd, hipStream_t s) {
  switch (dtype) {
    case 0: return conv_w<float>(p, bwd, s);
    case 1: return conv_w<bf16_t>(p, bwd, s);
    case 2: return conv_w<f16_t>(p, bwd, s);
    default: return conv_w<double>(p, bwd, s);
  }
}

}  // namespace ssm
