// The composed selective scan (models/scan.py:193-255) without its (B, L, D, N) tensors: one kernel
// per direction discretizes, scans with the chosen algorithm (tile_scan, ssm_tilescan.hpp) and
// contracts, where the reference materializes a, b, h, their gradients and the adjoint.
//
// A workgroup owns 64 / NP channels x NP states (one recurrence per lane) of one batch row and walks
// time in tiles of RL row lanes (wavefronts) x R steps; with the chunked algorithm, few workgroups and
// a long sequence it walks one segment of time (k_csc_sum).  Forward: a tile's x, delta, B, C are read
// while the previous tile is scanned, a and b are formed in registers as k_disc_fwd forms them, and
// y = sum_n C h is summed over the state lanes before it is stored.  It saves the state entering
// every tile.  Backward, from the last tile to the first: the tile's states are recomputed from the
// saved one with the same scan, lambda_t = dy_t C_t + a_{t+1} lambda_{t+1} is the same scan run
// against time with the adjoint mu = a lambda carried between tiles, and every gradient is formed
// from the registers with k_disc_bwd's arithmetic:
//   ddelta, dx   sums over the states, inside the wavefront
//   dBm, dCm     sums over the workgroup's channels inside the wavefront; one partial per tile of
//                channels, which k_csc_fin adds in float64, in a fixed order
//   dA           float64 running sums of 4-step float sums per lane, one partial per batch row
//                (and time segment)
//   dh0          the mu left at the first step
// All sums run in a fixed order, so results are bitwise reproducible.
//
// Bound: VALU issue (24 + 66 instructions per (b, t, d, n) element) and the latency of a tile's LDS
// exchanges, not HBM: the materialized form moved 6-8 (B, L, D, N) tensors forward and 19 in a
// training step, this moves 2 / CW of one (the dB / dC partials, CW = 64 / NP) twice.  B2 L2048
// D512 N16 float32, chunked, forward + backward: 41 + 87 + 11 us of kernels, 26 launches of 1,030 us
// before (sequential 51 + 97, Blelloch 47 + 86, Hillis-Steele 67 + 179).  8 steps per lane keep a
// backward lane's tile in registers (166 VGPRs: one workgroup per CU); 8 row lanes give the 256
// workgroups of that shape 2 wavefronts per SIMD.
#pragma once

#include "ssm_device.hpp"
#include "ssm_dpp.hpp"
#include "ssm_internal.hpp"
#include "ssm_tiles.hpp"
#include "ssm_tilescan.hpp"
#include "ssm_wave.hpp"

namespace ssm {

// ------------------------------------------------------------------ cross-lane sums
template <int CTRL> __device__ __forceinline__ float dpp_move(float v) { return dpp_f<CTRL>(v); }
template <int CTRL> __device__ __forceinline__ double dpp_move(double v) { return dpp_d<CTRL>(v); }

// Sums V values per lane over the lanes l ^ (a pattern flipping bit BIT, constant in the bits
// above it): while more than one value is left a lane keeps the half its bit selects and sends
// the other, so the lanes end up owning different values; the last value is added in place.
template <int CTRL, int BIT, int M, typename CT, int V>
__device__ __forceinline__ void fold_bit(CT (&v)[V], int lane) {
  if constexpr (M > 1) {
    const bool up = (lane >> BIT) & 1;
#pragma unroll
    for (int j = 0; j < M / 2; ++j) {
      const CT keep = up ? v[j + M / 2] : v[j], send = up ? v[j] : v[j + M / 2];
      v[j] = keep + dpp_move<CTRL>(send);
    }
  } else {
    v[0] += dpp_move<CTRL>(v[0]);
  }
}

constexpr int half_of(int m) { return m > 1 ? m / 2 : 1; }

// Sum of V values over a group of NP lanes (aligned): afterwards a lane owns the state_own values
// of index state_index(lane) + 0.., in v[0..).
template <int NP, int V> constexpr int state_own() { return V > (NP < 16 ? NP : 16) ? V / (NP < 16 ? NP : 16) : 1; }
template <int NP, typename CT, int V>
__device__ __forceinline__ void state_sum(CT (&v)[V], int lane) {
  constexpr int M2 = NP >= 16 ? half_of(V) : V, M1 = half_of(M2), M0 = half_of(M1);
  if constexpr (NP >= 16) fold_bit<0x140, 3, V>(v, lane);  // row_mirror
  fold_bit<0x141, 2, M2>(v, lane);                         // row_half_mirror
  fold_bit<0x4E, 1, M1>(v, lane);                          // quad_perm [2, 3, 0, 1]
  fold_bit<0xB1, 0, M0>(v, lane);                          // quad_perm [1, 0, 3, 2]
#pragma unroll
  for (int j = 0; j < state_own<NP, V>(); ++j) {
    if constexpr (NP >= 32) v[j] += __shfl_xor(v[j], 16);
    if constexpr (NP >= 64) v[j] += __shfl_xor(v[j], 32);
  }
}
template <int NP, int V>
__device__ __forceinline__ int state_index(int lane) {
  int m = V, idx = 0;
#pragma unroll
  for (int bit = NP >= 16 ? 3 : 2; bit >= 0; --bit) {
    if (m > 1) idx += (m /= 2) * ((lane >> bit) & 1);
  }
  return idx;
}
// Whether the lane is the one of its group that stores its values (several lanes of a group own
// the same ones when the group has more lanes than values).
template <int NP, int V>
__device__ __forceinline__ bool state_owner(int lane) {
  int m = V;
  bool own = true;
#pragma unroll
  for (int bit = NP >= 16 ? 3 : 2; bit >= 0; --bit) {
    if (m > 1) m /= 2;
    else own = own && !((lane >> bit) & 1);
  }
  return own && lane % NP < 16;
}

// a + b summed over the lanes l ^ 32 (ROW 0) or l ^ 16 (ROW 1): the lanes with the bit clear get
// a's sum, the others b's.
template <bool W32>
__device__ __forceinline__ void swap_words(unsigned &a, unsigned &b) {
  if constexpr (W32) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
  } else {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0];
    b = r[1];
  }
}
template <bool W32> __device__ __forceinline__ float swap_add(float a, float b) {
  unsigned x = __float_as_uint(a), y = __float_as_uint(b);
  swap_words<W32>(x, y);
  return __uint_as_float(x) + __uint_as_float(y);
}
template <bool W32> __device__ __forceinline__ double swap_add(double a, double b) {
  const unsigned long long x = __builtin_bit_cast(unsigned long long, a), y = __builtin_bit_cast(unsigned long long, b);
  unsigned xl = (unsigned)x, xh = (unsigned)(x >> 32), yl = (unsigned)y, yh = (unsigned)(y >> 32);
  swap_words<W32>(xl, yl);
  swap_words<W32>(xh, yh);
  return __builtin_bit_cast(double, ((unsigned long long)xh << 32) | xl) +
         __builtin_bit_cast(double, ((unsigned long long)yh << 32) | yl);
}
// Sum of V values over the wavefront's 64 / NP channels (the lanes of equal lane % NP); a lane then
// owns the V * NP / 64 values of index chan_index(lane) + 0.. .
template <int NP, typename CT, int V>
__device__ __forceinline__ void chan_sum(CT (&v)[V], int lane) {
  if constexpr (NP <= 32) {
#pragma unroll
    for (int j = 0; j < V / 2; ++j) v[j] = swap_add<true>(v[j], v[j + V / 2]);
  }
  if constexpr (NP <= 16) {
#pragma unroll
    for (int j = 0; j < V / 4; ++j) v[j] = swap_add<false>(v[j], v[j + V / 4]);
  }
  if constexpr (NP <= 8) {
    const bool up = (lane >> 3) & 1;
#pragma unroll
    for (int j = 0; j < V / 8; ++j) {
      const CT keep = up ? v[j + V / 8] : v[j], send = up ? v[j] : v[j + V / 8];
      v[j] = keep + dpp_move<0x128>(send);  // row_ror:8
    }
  }
}
template <int NP, int V>
__device__ __forceinline__ int chan_index(int lane) {
  int idx = 0;
  if (NP <= 32) idx += (lane >> 5) * (V / 2);
  if (NP <= 16) idx += ((lane >> 4) & 1) * (V / 4);
  if (NP <= 8) idx += ((lane >> 3) & 1) * (V / 8);
  return idx;
}

// ------------------------------------------------------------------ kernels
// Row lanes and steps per row lane of a tile.
template <typename CT, int ALGO> constexpr int cs_rl() { return csc_row_lanes(ALGO, sizeof(CT) == 8); }
template <typename CT, int ALGO> constexpr int cs_rows() { return csc_tile(ALGO, sizeof(CT) == 8) / cs_rl<CT, ALGO>(); }

// A wavefront's R steps x COLS channels (or states) of a (B, L, C) operand: read one element per lane
// along whichever axis has unit stride, and laid out in LDS as rows of R steps that a lane reads
// with 16-byte loads.  (A read per lane and step -- 4-5 R loads per tile of 64 or fewer distinct
// bytes each -- kept the address units 54 % busy: 62 + 121 us where this takes 41 + 87,
// at the shape above.)
template <typename CT, int R, int COLS>
struct TileIn {
  static constexpr int E = (R * COLS + kWave - 1) / kWave, RP = R + 16 / (int)sizeof(CT);
  const char *base;   // step 0, column c0 of batch row b
  int64_t s1;         // bytes between steps of the sequence
  uint32_t off[E];    // the lane's elements, below 2^31 bytes; kDropOffset (reads 0) for columns past the end
  bool tfast;
  __device__ __forceinline__ TileIn(const KView &v, int64_t b, int c0, int count, int step, int lane)
      : base((const char *)v.p + (b * v.s0 + c0 * v.s2) * (int64_t)sizeof(CT)), s1(v.s1 * (int64_t)sizeof(CT)),
        tfast(v.s1 == 1) {
#pragma unroll
    for (int i = 0; i < E; ++i) {
      int r, c;
      tc_of<R, COLS>(lane + i * kWave, tfast, r, c);
      const bool ok = lane + i * kWave < R * COLS && c0 + c < count;
      off[i] = ok ? (uint32_t)((r * step * v.s1 + c * v.s2) * (int64_t)sizeof(CT)) : kDropOffset;
    }
  }
  // Steps t0, t0 + step, ..; those at or past nv of the R read 0.
  __device__ __forceinline__ void load(CT (&v)[E], int t0, int nv, int lane) const {
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc((void *)(base + t0 * s1), (short)0, 0x7fffffff, kBufferFlags);
#pragma unroll
    for (int i = 0; i < E; ++i) {
      uint32_t o = off[i];
      if (nv < R) {  // uniform: only the ragged last tile
        int r, c;
        tc_of<R, COLS>(lane + i * kWave, tfast, r, c);
        o = r < nv ? o : kDropOffset;
      }
      v[i] = buf_load<CT>(rs, o);
    }
  }
  __device__ __forceinline__ void stage(CT (*S)[RP], const CT (&v)[E], int lane) const {
#pragma unroll
    for (int i = 0; i < E; ++i) {
      const int e = lane + i * kWave;
      int r, c;
      tc_of<R, COLS>(e, tfast, r, c);
      if (e < R * COLS) S[c][r] = v[i];
    }
  }
};

// The last row of each array stays zero: lanes of no channel or no state (pad lanes) read it, so that
// every one of their steps is the identity whatever the operands of the lanes beside them hold.  (The
// row is picked once; with B = C = 0 alone an infinite x, or a growing decay exp(-delta), gave 0 * inf.)
template <typename CT, int R, int NP, bool BWD>
struct StageLds {
  static constexpr int CW = kWave / NP, RP = R + 16 / (int)sizeof(CT);
  CT x[CW + 1][RP], dt[CW + 1][RP], g[BWD ? CW + 1 : 1][RP], B[NP + 1][RP], C[NP + 1][RP];
  __device__ __forceinline__ void clear_pad(int lane) {
    if (lane < RP) {
      x[CW][lane] = dt[CW][lane] = B[NP][lane] = C[NP][lane] = 0;
      if constexpr (BWD) g[CW][lane] = 0;
    }
  }
};

// A of -inf (-exp of a large A_log) as a finite value whose decay over any step is 0 too: the steps
// past the sequence's end have delta = 0, and 0 * inf is no identity.
template <typename CT>
__device__ __forceinline__ CT finite_decay(CT A) {
  const CT lim = sizeof(CT) == 8 ? (CT)-1e300 : (CT)-1e37;
  return A < lim ? lim : A;
}

// ------------------------------------------------------------------ time segments
// The chunked algorithm splits a long sequence over workgroups where its recurrences alone leave the GPU
// idle: k_csc_sum forms every segment's affine map (its decay product P and its end value E from
// zero), and each segment's walk first folds the maps of the segments before it.  In a segment a
// wavefront takes a contiguous eighth, without exchanges until the end.  BWD: the adjoint's map, against
// time (mu <- a (C dy + mu)).
template <typename CT, int NP, int METHOD, bool BWD>
__global__ void __launch_bounds__((cs_rl<CT, kChunk>() * kWave)) k_csc_sum(const CscParams p) {
  constexpr int RL = cs_rl<CT, kChunk>(), R = cs_rows<CT, kChunk>(), CW = kWave / NP;
  __shared__ __align__(16) StageLds<CT, R, NP, false> stage[RL];
  __shared__ CT sP[RL][kWave], sE[RL][kWave];
  const int lane = threadIdx.x % kWave, tr = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  StageLds<CT, R, NP, false> &S = stage[tr];
  const int c = lane / NP, n = lane % NP, d0 = blockIdx.x * CW, d = d0 + c;
  const int64_t b = blockIdx.y;
  const int L = (int)p.L, D = (int)p.D, N = (int)p.N;
  const bool valid = d < D && n < N;
  const AConst<CT> ac = make_aconst(valid ? finite_decay(vload<CT>(p.A, d * p.A.s0 + n * p.A.s1)) : (CT)-1);
  const int cr = valid ? c : CW, nr = valid ? n : NP;
  const TileIn<CT, R, CW> iu(BWD ? p.dy : p.x, b, d0, D, 1, lane), id(p.dt, b, d0, D, 1, lane);
  const TileIn<CT, R, NP> iV(BWD ? p.Cm : p.Bm, b, 0, N, 1, lane);
  const int seg = (int)blockIdx.z + (BWD ? 1 : 0);  // nothing follows the last segment, or the adjoint's first
  const int w0 = (seg * p.seg_tiles * RL + tr * p.seg_tiles) * R, w1 = min(w0 + p.seg_tiles * R, L);
  CT nu[iu.E], nd[id.E], nV[iV.E];
  auto fetch = [&](int k) {
    const int t0 = w0 + k * R, nv = L - t0;
    iu.load(nu, t0, nv, lane);
    id.load(nd, t0, nv, lane);
    iV.load(nV, t0, nv, lane);
  };
  const int nb = w0 < w1 ? (w1 - w0 + R - 1) / R : 0;  // the same for the whole wavefront
  CT P = 1, E = 0;
  S.clear_pad(lane);
  if (nb > 0) fetch(BWD ? nb - 1 : 0);
  for (int k = 0; k < nb; ++k) {
    iu.stage(S.x, nu, lane);
    id.stage(S.dt, nd, lane);
    iV.stage(S.B, nV, lane);
    wave_lds_sync();
    if (k + 1 < nb) fetch(BWD ? nb - 2 - k : k + 1);
    CT dt[R], u[R], V[R];
    lds_row(&S.dt[cr][0], dt);
    lds_row(&S.x[cr][0], u);
    lds_row(&S.B[nr][0], V);
#pragma unroll
    for (int q = 0; q < R; ++q) {  // a zero step is the identity
      const int r = BWD ? R - 1 - q : q;
      CT a, coef;
      disc<METHOD>(dt[r], ac, a, coef);
      if constexpr (BWD) E = a * fma(V[r], u[r], E);
      else E = fma(a, E, bcoef<METHOD>(dt[r], coef) * (V[r] * u[r]));
      P *= a;
    }
    wave_lds_sync();
  }
  sP[tr][lane] = P;
  sE[tr][lane] = E;
  lds_barrier();
  if (tr == 0 && valid) {
    P = 1;
    E = 0;
#pragma unroll
    for (int q = 0; q < RL; ++q) {
      const int k = BWD ? RL - 1 - q : q;
      E = fma(sP[k][lane], E, sE[k][lane]);
      P *= sP[k][lane];
    }
    CT *const ws = (CT *)p.ws_seg;
    const int64_t o = ((b * p.nseg + seg) * p.D + d) * p.N + n;
    ws[o] = P;
    ws[p.B * p.nseg * p.D * p.N + o] = E;
  }
}

// v through the maps of `count` segments, the first at s0 and each following `dir` further; 8 are read
// at a time (clamped to the last), the same folds in every wavefront of a workgroup.
template <typename CT>
__device__ __forceinline__ CT seg_fold(const CscParams &p, int64_t b, int d, int n, int s0, int dir, int count, CT v) {
  const int64_t plane = p.D * p.N, half = p.B * p.nseg * plane;
  const CT *const ws = (const CT *)p.ws_seg + b * p.nseg * plane + (int64_t)d * p.N + n;
  for (int k = 0; k < count; k += 8) {
    CT P[8], E[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int64_t o = (s0 + dir * min(k + j, count - 1)) * plane;
      P[j] = ws[o];
      E[j] = ws[half + o];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (k + j < count) v = fma(P[j], v, E[j]);
  }
  return v;
}

// ------------------------------------------------------------------ the walks
template <typename CT, int NP, int METHOD, int ALGO, bool SEG>
__global__ void __launch_bounds__((cs_rl<CT, ALGO>() * kWave)) k_csc_fwd(const CscParams p) {
  constexpr int RL = cs_rl<CT, ALGO>(), R = cs_rows<CT, ALGO>(), T = RL * R, CW = kWave / NP;
  constexpr int ST = ALGO == kHs ? RL : 1;  // steps between a row lane's consecutive ones
  __shared__ TileLds<CT, ALGO, RL, R> X;
  __shared__ __align__(16) StageLds<CT, R, NP, false> stage[RL];
  const int lane = threadIdx.x % kWave, tr = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  StageLds<CT, R, NP, false> &S = stage[tr];
  const int c = lane / NP, n = lane % NP, d0 = xcd_tile() * CW, d = d0 + c;
  const int64_t b = blockIdx.y;
  const int L = (int)p.L, D = (int)p.D, N = (int)p.N;
  const bool valid = d < D && n < N;
  const AConst<CT> ac = make_aconst(valid ? finite_decay(vload<CT>(p.A, d * p.A.s0 + n * p.A.s1)) : (CT)-1);
  const int cr = valid ? c : CW, nr = valid ? n : NP;  // rows of the staged operands
  const TileIn<CT, R, CW> ix(p.x, b, d0, D, ST, lane), id(p.dt, b, d0, D, ST, lane);
  const TileIn<CT, R, NP> iB(p.Bm, b, 0, N, ST, lane), iC(p.Cm, b, 0, N, ST, lane);
  CT carry = p.h0.p && valid ? vload<CT>(p.h0, b * p.h0.s0 + d * p.h0.s1 + n * p.h0.s2) : (CT)0;
  CT nx[ix.E], nd[id.E], nB[iB.E], nC[iC.E];
  auto fetch = [&](int base) {  // steps past the end and padded channels and states read zeros
    const int t0 = base + tile_step<ALGO, RL, R>(tr, 0), nv = t0 < L ? (L - t0 + ST - 1) / ST : 0;
    ix.load(nx, t0, nv, lane);
    id.load(nd, t0, nv, lane);
    iB.load(nB, t0, nv, lane);
    iC.load(nC, t0, nv, lane);
  };
  const int seg = SEG ? (int)blockIdx.z : 0, first = SEG ? seg * p.seg_tiles : 0;
  const int end = SEG ? min(L, (first + p.seg_tiles) * T) : L;
  fetch(first * T);
  S.clear_pad(lane);
  if (SEG && valid) carry = seg_fold<CT>(p, b, d, n, 0, 1, seg, carry);
  int buf = 0, i = first;
  const int yi = state_index<NP, R>(lane);
  const bool yown = state_owner<NP, R>(lane) && d < D;
  for (int base = first * T; base < end; base += T, ++i) {
    if (p.saved.p && tr == 0 && valid)
      ((CT *)p.saved.p)[b * p.saved.s0 + i * p.saved.s1 + d * p.saved.s2 + n] = carry;
    ix.stage(S.x, nx, lane);
    id.stage(S.dt, nd, lane);
    iB.stage(S.B, nB, lane);
    iC.stage(S.C, nC, lane);
    wave_lds_sync();
    if (base + T < end) fetch(base + T);
    CT a[R], h[R], y[R], x[R], dt[R], Bv[R];
    lds_row(&S.dt[cr][0], dt);
    lds_row(&S.x[cr][0], x);
    lds_row(&S.B[nr][0], Bv);
    lds_row(&S.C[nr][0], y);
#pragma unroll
    for (int r = 0; r < R; ++r) {  // a zero step is the identity
      CT coef;
      disc<METHOD>(dt[r], ac, a[r], coef);
      h[r] = bcoef<METHOD>(dt[r], coef) * (Bv[r] * x[r]);
    }
    CT hin;
    tile_scan<CT, ALGO, RL, R>(X, a, h, carry, hin, tr, lane, buf);
#pragma unroll
    for (int r = 0; r < R; ++r) y[r] *= h[r];
    state_sum<NP>(y, lane);
#pragma unroll
    for (int j = 0; j < state_own<NP, R>(); ++j) {
      const int t = base + tile_step<ALGO, RL, R>(tr, yi + j);
      if (yown && t < L) vstore<CT>(p.y, b * p.y.s0 + t * p.y.s1 + d * p.y.s2, y[j]);
    }
    wave_lds_sync();
  }
  if (p.last.p && end == L && tr == 0 && valid) vstore<CT>(p.last, b * p.last.s0 + d * p.last.s1 + n * p.last.s2, carry);
}

template <typename CT, int NP, int METHOD, int ALGO, bool SEG>
__global__ void __launch_bounds__((cs_rl<CT, ALGO>() * kWave)) k_csc_bwd(const CscParams p) {
  constexpr int RL = cs_rl<CT, ALGO>(), R = cs_rows<CT, ALGO>(), T = RL * R, CW = kWave / NP, V = 2 * R;
  constexpr int ST = ALGO == kHs ? RL : 1;
  __shared__ TileLds<CT, ALGO, RL, R> X;
  __shared__ __align__(16) StageLds<CT, R, NP, true> stage[RL];
  __shared__ CT a0s[RL][kWave];      // the row lanes' first decay (consecutive steps)
  __shared__ double red[RL][kWave];  // dA of the row lanes
  const int lane = threadIdx.x % kWave, tr = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  StageLds<CT, R, NP, true> &S = stage[tr];
  const int c = lane / NP, n = lane % NP, tile = xcd_tile(), d0 = tile * CW, d = d0 + c;
  const int64_t b = blockIdx.y;
  const int L = (int)p.L, D = (int)p.D, N = (int)p.N;
  const bool valid = d < D && n < N;
  const AConst<CT> ac = make_aconst(valid ? finite_decay(vload<CT>(p.A, d * p.A.s0 + n * p.A.s1)) : (CT)-1);
  const int cr = valid ? c : CW, nr = valid ? n : NP;  // rows of the staged operands
  const TileIn<CT, R, CW> ix(p.x, b, d0, D, ST, lane), id(p.dt, b, d0, D, ST, lane), ig(p.dy, b, d0, D, ST, lane);
  const TileIn<CT, R, NP> iB(p.Bm, b, 0, N, ST, lane), iC(p.Cm, b, 0, N, ST, lane);
  // mu: the adjoint entering the tile's last step from the steps after it
  CT mu = p.dlast.p && valid ? vload<CT>(p.dlast, b * p.dlast.s0 + d * p.dlast.s1 + n * p.dlast.s2) : (CT)0;
  CT nx[ix.E], nd[id.E], ng[ig.E], nB[iB.E], nC[iC.E], nh = 0;
  auto fetch = [&](int i) {
    const int t0 = i * T + tile_step<ALGO, RL, R>(tr, 0), nv = t0 < L ? (L - t0 + ST - 1) / ST : 0;
    ix.load(nx, t0, nv, lane);
    id.load(nd, t0, nv, lane);
    ig.load(ng, t0, nv, lane);
    iB.load(nB, t0, nv, lane);
    iC.load(nC, t0, nv, lane);
    if (valid) nh = ((const CT *)p.saved.p)[b * p.saved.s0 + i * p.saved.s1 + d * p.saved.s2 + n];
  };
  const int seg = SEG ? (int)blockIdx.z : 0, first = SEG ? seg * p.seg_tiles : 0;
  const int all = (L + T - 1) / T, nt = SEG ? min(all, first + p.seg_tiles) : all;  // tiles first .. nt - 1
  fetch(nt - 1);
  S.clear_pad(lane);
  if (SEG && valid) mu = seg_fold<CT>(p, b, d, n, p.nseg - 1, -1, p.nseg - 1 - seg, mu);
  int buf = 0;
  double gA = 0;
  const int oi = state_index<NP, V>(lane), wi = chan_index<NP, V>(lane);
  const bool own = state_owner<NP, V>(lane) && d < D;
  CT *const ws = (CT *)p.ws_bc + (b * p.ntiles + tile) * p.L * 2 * NP;  // (L, {B, C}, NP) partials
  for (int i = nt - 1; i >= first; --i) {
    const int base = i * T;
    CT hc = nh;  // the state entering the tile
    const CT hc0 = hc;
    ix.stage(S.x, nx, lane);
    id.stage(S.dt, nd, lane);
    ig.stage(S.g, ng, lane);
    iB.stage(S.B, nB, lane);
    iC.stage(S.C, nC, lane);
    wave_lds_sync();
    if (i > first) fetch(i - 1);
    CT a[R], a0[R], coef[R], h[R], dt[R], x[R], Bv[R], dy[R], g[R];
    lds_row(&S.dt[cr][0], dt);
    lds_row(&S.x[cr][0], x);
    lds_row(&S.B[nr][0], Bv);
    lds_row(&S.g[cr][0], dy);
    lds_row(&S.C[nr][0], g);
#pragma unroll
    for (int r = 0; r < R; ++r) {  // a zero step is the identity
      g[r] *= dy[r];
      disc<METHOD>(dt[r], ac, a[r], coef[r]);
      a0[r] = a[r];
      h[r] = bcoef<METHOD>(dt[r], coef[r]) * (Bv[r] * x[r]);
    }
    if constexpr (ALGO != kHs) a0s[tr][lane] = a0[0];
    CT hin, hp[R], m[R], afirst;
    tile_scan<CT, ALGO, RL, R>(X, a, h, hc, hin, tr, lane, buf);
    // the state before each step and the decay of the step after it (1 past the tile: mu already
    // carries that decay)
    if constexpr (ALGO == kHs) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        X.A[buf][tr + RL * r][lane] = a0[r];
        X.S[buf][tr + RL * r][lane] = h[r];
      }
      lds_barrier();
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int k = tr + RL * r;
        hp[r] = k > 0 ? X.S[buf][k > 0 ? k - 1 : 0][lane] : hc0;
        m[R - 1 - r] = k + 1 < T ? X.A[buf][k + 1 < T ? k + 1 : k][lane] : (CT)1;
      }
      afirst = X.A[buf][0][lane];
      buf ^= 1;
    } else {
      const CT an = a0s[tr + 1 < RL ? tr + 1 : tr][lane];
      afirst = a0s[0][lane];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        hp[r] = r > 0 ? h[r > 0 ? r - 1 : 0] : hin;
        m[R - 1 - r] = r + 1 < R ? a0[r + 1 < R ? r + 1 : r] : (tr + 1 < RL ? an : (CT)1);
      }
    }
    // the adjoint: the same scan against time
    CT lam[R];
#pragma unroll
    for (int r = 0; r < R; ++r) lam[R - 1 - r] = g[r];
    tile_scan<CT, ALGO, RL, R>(X, m, lam, mu, hin, RL - 1 - tr, lane, buf);
    mu *= afirst;
    CT v[V], w[V], gA4 = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const CT l = lam[R - 1 - r];
      CT dadz, dbdd, d2f;
      dfactors<METHOD>(dt[r], ac, a0[r], coef[r], dadz, dbdd, d2f);
      const CT bx = Bv[r] * x[r], gz = (l * hp[r]) * dadz, gbc = l * bcoef<METHOD>(dt[r], coef[r]);
      v[r] = gbc * Bv[r];
      v[R + r] = fma(ac.A, gz, l * dbdd * bx);
      gA4 += fma(dt[r], gz, l * d2f * bx);
      w[r] = gbc * x[r];
      w[R + r] = dy[r] * h[r];
      if (r % 4 == 3) {
        gA += (double)gA4;
        gA4 = 0;
      }
    }
    state_sum<NP>(v, lane);
#pragma unroll
    for (int j = 0; j < state_own<NP, V>(); ++j) {
      const int q = (oi + j) / R, t = base + tile_step<ALGO, RL, R>(tr, (oi + j) % R);
      if (own && t < L) {
        if (q == 0) vstore<CT>(p.dx, b * p.dx.s0 + t * p.dx.s1 + d * p.dx.s2, v[j]);
        else vstore<CT>(p.ddelta, b * p.ddelta.s0 + t * p.ddelta.s1 + d * p.ddelta.s2, v[j]);
      }
    }
    chan_sum<NP>(w, lane);
#pragma unroll
    for (int j = 0; j < V / CW; ++j) {
      const int q = (wi + j) / R, t = base + tile_step<ALGO, RL, R>(tr, (wi + j) % R);
      if (t < L) ws[((int64_t)t * 2 + q) * NP + n] = w[j];
    }
    wave_lds_sync();
  }
  red[tr][lane] = gA;
  lds_barrier();
  if (tr == 0 && valid) {
    double s = 0;
#pragma unroll
    for (int q = 0; q < RL; ++q) s += red[q][lane];
    ((double *)p.ws_dA)[((SEG ? b * p.nseg + seg : b) * p.D + d) * p.N + n] = s;
    if (p.dh0.p && seg == 0) vstore<CT>(p.dh0, b * p.dh0.s0 + d * p.dh0.s1 + n * p.dh0.s2, mu);
  }
}

template <typename CT, int NP, int METHOD, int ALGO, bool SEG>
static hipError_t csc_t(const CscParams &p, bool bwd, hipStream_t s) {
  constexpr int CW = kWave / NP;
  const unsigned tiles = (unsigned)((p.D + CW - 1) / CW), threads = cs_rl<CT, ALGO>() * kWave;
  if constexpr (SEG) {
    const dim3 g(tiles, (unsigned)p.B, (unsigned)p.nseg - 1);
    if (bwd) hipLaunchKernelGGL((k_csc_sum<CT, NP, METHOD, true>), g, dim3(threads), 0, s, p);
    else hipLaunchKernelGGL((k_csc_sum<CT, NP, METHOD, false>), g, dim3(threads), 0, s, p);
  }
  const dim3 grid(tiles, (unsigned)p.B, (unsigned)p.nseg);
  if (bwd) hipLaunchKernelGGL((k_csc_bwd<CT, NP, METHOD, ALGO, SEG>), grid, dim3(threads), 0, s, p);
  else hipLaunchKernelGGL((k_csc_fwd<CT, NP, METHOD, ALGO, SEG>), grid, dim3(threads), 0, s, p);
  return hipGetLastError();
}

template <typename CT, int NP, int ALGO, bool SEG>
static hipError_t csc_m(const CscParams &p, int method, bool bwd, hipStream_t s) {
  return method == 0 ? csc_t<CT, NP, 0, ALGO, SEG>(p, bwd, s) : method == 1 ? csc_t<CT, NP, 1, ALGO, SEG>(p, bwd, s)
                                                                       : csc_t<CT, NP, 2, ALGO, SEG>(p, bwd, s);
}

template <typename CT, int ALGO, bool SEG>
static hipError_t csc_n(const CscParams &p, int method, int np, bool bwd, hipStream_t s) {
  switch (np) {
    case 8: return csc_m<CT, 8, ALGO, SEG>(p, method, bwd, s);
    case 16: return csc_m<CT, 16, ALGO, SEG>(p, method, bwd, s);
    case 32: return csc_m<CT, 32, ALGO, SEG>(p, method, bwd, s);
    default: return csc_m<CT, 64, ALGO, SEG>(p, method, bwd, s);
  }
}

template <int ALGO, bool SEG>
hipError_t launch_csc_algo(const CscParams &p, int dtype, int method, int np, bool bwd, hipStream_t s) {
  return dtype == 3 ? csc_n<double, ALGO, SEG>(p, method, np, bwd, s) : csc_n<float, ALGO, SEG>(p, method, np, bwd, s);
}

}  // namespace ssm
