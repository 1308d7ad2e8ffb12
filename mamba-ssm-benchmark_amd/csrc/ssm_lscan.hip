// Linear-recurrence scan algorithms for gfx950: h_t = a_t h_{t-1} + b_t over (B, L, M).
//
// Replaces the four torch scans of models/scan.py with kernels that keep each algorithm's
// structure (so `scan=` still selects an algorithm, as in the reference's SCANS registry,
// models/scan.py:168-173).  One walk serves all four (k_lscan_walk): a workgroup owns 64
// neighbouring recurrences (lanes along m, so every global access is coalesced) and walks time
// in tiles; row lane tr, a wavefront, holds its steps of the tile in registers while the next
// tile's are read.  What the tile does with them is the algorithm:
//   sequential     models/scan.py:70-76    the row lanes take turns, each walking its 16 steps
//                                          from the state the previous one hands over; forward
//                                          passes of short or wide scans run one wavefront per
//                                          workgroup instead (k_lscan_seqt).
//   hillis_steele  models/scan.py:87-98    recursive doubling along the tile (offsets below the
//                                          row lanes through LDS, the others in registers); the
//                                          state entering a tile is folded into its first
//                                          element (as _fold_h0 does with h0, :79-84).
//   blelloch       models/scan.py:101-135  up-sweep / down-sweep along the tile (a lane's
//                                          16-step block in registers, the block roots through
//                                          LDS), giving exclusive (A, S) prefixes;
//                                          h = a (A h_in + S) + b, the tile's last h carried.
//   chunked        models/scan.py:142-165  a row lane's 16 steps are a chunk: its summary
//                                          (P = prod a, E = end state from zero) goes through
//                                          LDS, the state entering every chunk is folded from
//                                          the summaries before it, and the chunk is scanned
//                                          from that state.  With too few recurrences to fill
//                                          the GPU the chunks are spread over it instead, in
//                                          three launches: summaries, a scan over them per
//                                          (b, m), then each chunk scanned from its entering
//                                          state.
// Direction: with `reverse` the recurrence runs from t = L-1 down to 0.  With `shift` (used
// by the adjoint) the multiplier at a step is the a of the previous step in processing order
// and 1 for the first step: lambda_t = g_t + a_{t+1} lambda_{t+1} (models/scan.py:239-240); the
// adjoint's da and dh0 (:242-248) are formed where lambda is stored.
//
// Bound: HBM.  3 (adjoint: 5) tensors of s B L M bytes move once.  What a workgroup keeps in
// flight sets the rate: 8 row lanes x 16 steps x 2-3 tensors x 256 bytes.  At (B, L, M) = (2,
// 4096, 8192) float32, forward + adjoint, where a copy of the same bytes takes 155 + 259 us:
// chunked 159 + 257 us (in three launches with a separate adjoint epilogue 295 + 570), blelloch
// 159 + 256 (with 4 row lanes 200 + 484), hillis_steele 181 + 269 (237 + 511), sequential 156 +
// 256 (one wavefront per workgroup 185 + 467).
#include <algorithm>

#include "ssm_device.hpp"
#include "ssm_dpp.hpp"
#include "ssm_internal.hpp"
#include "ssm_tiles.hpp"
#include "ssm_tilescan.hpp"
#include "ssm_wave.hpp"

namespace ssm {

template <typename CT>
struct Chain {
  const LscanParams &P;
  int64_t b, m;
  __device__ __forceinline__ int t_of(int pos) const { return P.reverse ? (int)P.L - 1 - pos : pos; }
  __device__ __forceinline__ CT a_at(int t) const {
    return vload<CT>(P.a, b * P.a.s0 + (int64_t)t * P.a.s1 + m * P.a.s2);
  }
  // multiplier used at processing position pos
  __device__ __forceinline__ CT mult(int pos) const {
    if (!P.shift) return a_at(t_of(pos));
    return pos > 0 ? a_at(t_of(pos - 1)) : (CT)1;
  }
  __device__ __forceinline__ CT b_at(int t) const {
    return vload<CT>(P.b, b * P.b.s0 + (int64_t)t * P.b.s1 + m * P.b.s2);
  }
  __device__ __forceinline__ int64_t h_off(int t) const { return b * P.h.s0 + (int64_t)t * P.h.s1 + m * P.h.s2; }
  // Adjoint (GRAD): the forward scan's state before the step at processing position pos -- the
  // state at the next position, since the adjoint runs against the forward scan; read at a clamped
  // position, so that h0f() (read once, not in the walk) can take its place at the last one.
  __device__ __forceinline__ CT hprev_at(int pos) const {
    return vload<CT>(P.hf, b * P.hf.s0 + (int64_t)t_of(min(pos + 1, (int)P.L - 1)) * P.hf.s1 + m * P.hf.s2);
  }
  __device__ __forceinline__ CT h0f() const {
    return P.h0f.p ? vload<CT>(P.h0f, b * P.h0f.s0 + m * P.h0f.s1) : (CT)0;
  }
  // Stores the scan's value v at position pos; with GRAD, v is lambda (= db) and da = lambda
  // h_{prev} goes out with it.
  template <bool GRAD>
  __device__ __forceinline__ void put(int pos, CT v, CT hp) const {
    const int t = t_of(pos);
    vstore<CT>(P.h, h_off(t), v);
    if constexpr (GRAD) vstore<CT>(P.da, b * P.da.s0 + (int64_t)t * P.da.s1 + m * P.da.s2, v * hp);
  }
  // dh0 = a lambda of the last position (the forward scan's first step).
  __device__ __forceinline__ void put_dh0(CT v) const {
    if (P.dh0.p) vstore<CT>(P.dh0, b * P.dh0.s0 + m * P.dh0.s1, a_at(t_of((int)P.L - 1)) * v);
  }
  __device__ __forceinline__ CT h0() const {
    return P.h0.p ? vload<CT>(P.h0, b * P.h0.s0 + m * P.h0.s1) : (CT)0;
  }
};

// ------------------------------------------------------------------ the tiled walk
// Steps per row lane and tile (Hillis-Steele keeps every step of a tile in LDS twice).
constexpr int scan_rows(int algo) { return algo == kHs ? 8 : 16; }

template <typename CT, int ALGO, int RL, bool GRAD>
__global__ void __launch_bounds__(RL * kScanMC) k_lscan_walk(const LscanParams P) {
  constexpr int R = scan_rows(ALGO), T = RL * R;
  static_assert(kScanMC == kWave, "a row lane is a wavefront");
  __shared__ TileLds<CT, ALGO, RL, R> X;
  const int mi = threadIdx.x % kScanMC, tr = __builtin_amdgcn_readfirstlane(threadIdx.x / kScanMC);
  const int64_t m = (int64_t)blockIdx.x * kScanMC + mi;
  const bool mval = m < P.M;
  Chain<CT> ch{P, (int64_t)blockIdx.y, mval ? m : P.M - 1};
  const int L = (int)P.L;
  auto step = [&](int r) { return tile_step<ALGO, RL, R>(tr, r); };
  CT carry = ch.h0();
  const CT hfirst = GRAD ? ch.h0f() : (CT)0;
  CT na[R] = {}, nb[R] = {}, nh[GRAD ? R : 1] = {};
  auto read = [&](int pos, int r) {
    na[r] = ch.mult(pos);
    nb[r] = ch.b_at(ch.t_of(pos));
    if constexpr (GRAD) nh[r] = ch.hprev_at(pos);
  };
  // A row lane past the end of the sequence reads nothing; at the end, one of consecutive steps reads at
  // clamped positions (a second copy of the reads for whole tiles costs a short scan more than it
  // saves), Hillis-Steele's skip theirs one by one (half a last tile of theirs lies past the end: L 80,
  // 512 workgroups, forward 11.9 -> 11.0 us).  All conditions are uniform over the wavefront.
  auto fetch = [&](int base) {
    if (base + step(0) >= L) return;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if constexpr (ALGO == kHs) {
        if (base + step(r) < L) read(base + step(r), r);
      } else {
        read(min(base + step(r), L - 1), r);
      }
    }
  };
  fetch(0);
  int buf = 0;
  for (int base = 0; base < L; base += T) {
    CT a[R], b[R], hp[GRAD ? R : 1];
#pragma unroll
    for (int r = 0; r < R; ++r) {  // a position past the end is the identity (1, 0)
      const bool in = base + step(r) < L;
      a[r] = in ? na[r] : (CT)1;
      b[r] = in ? nb[r] : (CT)0;
      if constexpr (GRAD) hp[r] = base + step(r) + 1 < L ? nh[r] : hfirst;
    }
    if (base + T < L) fetch(base + T);
    CT hin;
    auto emit = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int pos = base + step(r);
        if (mval && pos < L) ch.template put<GRAD>(pos, b[r], hp[GRAD ? r : 0]);
        if (GRAD && mval && pos + 1 == L) ch.put_dh0(b[r]);
      }
    };
    tile_scan<CT, ALGO, RL, R>(X, a, b, carry, hin, tr, mi, buf, emit);
  }
}

// ------------------------------------------------------------------ sequential, one wavefront
// Sequential, forward, float, unit stride along m.  A wavefront owns 64 consecutive recurrences m of one
// batch row and walks 16-step blocks.  A block's a and b tiles (16 steps x 64 recurrences) are read
// with 16-byte loads -- a lane reads 4 recurrences of one step, so one load instruction carries 4
// steps where a read per recurrence carries one -- and transposed through LDS so that each lane
// walks its own recurrence; the block's states go back through LDS and leave as 16-byte stores.
// Reads run kSeqTAhead blocks ahead, at clamped positions (past the end: re-reads of the last step,
// never used).
constexpr int kSeqTB = 16, kSeqTAhead = 3;
typedef float f32x4 __attribute__((ext_vector_type(4)));  // a native vector (HIP's float4 is a struct)

__global__ void __launch_bounds__(64) k_lscan_seqt(const LscanParams P) {
  __shared__ __align__(16) float sA[kSeqTB][64], sB[kSeqTB][64], sH[kSeqTB][64];
  const int lane = threadIdx.x;
  const int64_t b = blockIdx.y, m0 = (int64_t)blockIdx.x * 64;
  const int L = (int)P.L;
  const int rl = lane / 16, cl = (lane % 16) * 4;  // the lane's row in a group of 4 steps, its column
  Chain<float> ch{P, b, m0 + lane};
  float h = ch.h0();
  const float *pa = (const float *)P.a.p + b * P.a.s0 + m0 + cl;
  const float *pb = (const float *)P.b.p + b * P.b.s0 + m0 + cl;
  float *ph = (float *)P.h.p + b * P.h.s0 + m0 + cl;
  struct Blk {
    f32x4 a[kSeqTB / 4], b[kSeqTB / 4];
  };
  auto fetch = [&](Blk &k, int pos0) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < kSeqTB / 4; ++j) {
      const int64_t t = ch.t_of(min(pos0 + rl + 4 * j, L - 1));
      k.a[j] = *(const f32x4 *)(pa + t * P.a.s1);
      k.b[j] = *(const f32x4 *)(pb + t * P.b.s1);
    }
  };
  auto run = [&](const Blk &k, int pos0) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < kSeqTB / 4; ++j) {
      *(f32x4 *)&sA[rl + 4 * j][cl] = k.a[j];
      *(f32x4 *)&sB[rl + 4 * j][cl] = k.b[j];
    }
    wave_lds_sync();
#pragma unroll
    for (int r = 0; r < kSeqTB; ++r) {
      h = fmaf(sA[r][lane], h, sB[r][lane]);
      sH[r][lane] = h;
    }
    wave_lds_sync();
#pragma unroll
    for (int j = 0; j < kSeqTB / 4; ++j) {
      const int pos = pos0 + rl + 4 * j;
      const f32x4 v = *(const f32x4 *)&sH[rl + 4 * j][cl];
      if (pos < L) *(f32x4 *)(ph + (int64_t)ch.t_of(pos) * P.h.s1) = v;
    }
    wave_lds_sync();  // the next block's tiles reuse the LDS
  };
  Blk k[kSeqTAhead];
  static_for<0, kSeqTAhead>([&](auto icst) { fetch(k[decltype(icst)::value], decltype(icst)::value * kSeqTB); });
  for (int pos = 0; pos < L; pos += kSeqTAhead * kSeqTB) {
    // blocks past the end are skipped (their reads, clamped, are never used)
    static_for<0, kSeqTAhead>([&](auto icst) {
      constexpr int i = decltype(icst)::value;
      if (pos + i * kSeqTB < L) run(k[i], pos + i * kSeqTB);
      fetch(k[i], pos + (i + kSeqTAhead) * kSeqTB);
    });
  }
}

// ------------------------------------------------------------------ chunked (three phases)
// Reduce, carry, scan: each chunk's summary (P = product of its multipliers, E = its end
// state from zero) is formed without writing any state; a sequential scan over the summaries
// gives every chunk's entering state h_in; each chunk is then scanned from h_in.  The chunks'
// states equal scan_chunked's local states corrected by P_t h_in (models/scan.py:152-164),
// to rounding, and the states are written once instead of written, re-read and rewritten.
constexpr int kSeqAhead = 16;  // steps whose inputs are read before their dependent updates

// Walks positions [p0, p1) of a chain from state h: h <- mult h + b at each step, with the
// product of the multipliers in prod (REDUCE) or every state stored (otherwise).
template <typename CT, bool REDUCE, bool GRAD>
__device__ __forceinline__ void chunk_walk(const LscanParams &P, const Chain<CT> &ch, int p0, int p1, CT &h,
                                           CT &prod) {
  const bool last = GRAD && p1 == (int)P.L;
  const CT hfirst = last ? ch.h0f() : (CT)0;
  int pos = p0;
  for (; pos + kSeqAhead <= p1; pos += kSeqAhead) {  // inputs read ahead of the updates
    CT av[kSeqAhead], bv[kSeqAhead], hp[GRAD ? kSeqAhead : 1];
#pragma unroll
    for (int u = 0; u < kSeqAhead; ++u) {
      av[u] = ch.mult(pos + u);
      bv[u] = ch.b_at(ch.t_of(pos + u));
      if constexpr (GRAD) hp[u] = ch.hprev_at(pos + u);
    }
#pragma unroll
    for (int u = 0; u < kSeqAhead; ++u) {
      h = fma(av[u], h, bv[u]);
      if constexpr (REDUCE) prod *= av[u];
      else ch.template put<GRAD>(pos + u, h, last && pos + u + 1 == p1 ? hfirst : hp[GRAD ? u : 0]);
    }
  }
  for (; pos < p1; ++pos) {
    const CT a = ch.mult(pos);
    h = fma(a, h, ch.b_at(ch.t_of(pos)));
    if constexpr (REDUCE) prod *= a;
    else ch.template put<GRAD>(pos, h, !GRAD ? (CT)0 : last && pos + 1 == p1 ? hfirst : ch.hprev_at(pos));
  }
  if constexpr (GRAD && !REDUCE) {
    if (last) ch.put_dh0(h);
  }
}

template <typename CT>
__global__ void __launch_bounds__(256) k_lscan_chunk_reduce(const LscanParams P) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= P.B * P.nc * P.M) return;
  const int64_t m = i % P.M, cj = (i / P.M) % P.nc, b = i / (P.M * P.nc);
  Chain<CT> ch{P, b, m};
  const int p0 = (int)cj * P.chunk;
  const int p1 = p0 + P.chunk < (int)P.L ? p0 + P.chunk : (int)P.L;
  CT h = 0, prod = 1;
  chunk_walk<CT, true, false>(P, ch, p0, p1, h, prod);
  CT *ws = (CT *)P.ws;
  const int64_t stride = P.B * P.nc * P.M;
  ws[i] = prod;        // P: product of the chunk's multipliers
  ws[stride + i] = h;  // E: end state from zero
}

template <typename CT>
__global__ void __launch_bounds__(256) k_lscan_chunk_carry(const LscanParams P) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= P.B * P.M) return;
  const int64_t m = i % P.M, b = i / P.M;
  Chain<CT> ch{P, b, m};
  CT *ws = (CT *)P.ws;
  const int64_t stride = P.B * P.nc * P.M;
  CT hin = ch.h0();
  // the summaries of kCarryGroup chunks are read together (unconditionally: a clamped chunk is
  // never used), then folded in order
  for (int c0 = 0; c0 < P.nc; c0 += kCarryGroup) {
    CT Pv[kCarryGroup], Ev[kCarryGroup];
#pragma unroll
    for (int j = 0; j < kCarryGroup; ++j) {
      const int64_t k = (b * P.nc + min((int64_t)(c0 + j), P.nc - 1)) * P.M + m;
      Pv[j] = ws[k];
      Ev[j] = ws[stride + k];
    }
#pragma unroll
    for (int j = 0; j < kCarryGroup; ++j) {
      if (c0 + j < P.nc) {
        ws[2 * stride + (b * P.nc + c0 + j) * P.M + m] = hin;  // state entering chunk c0 + j
        hin = fma(Pv[j], hin, Ev[j]);
      }
    }
  }
}

template <typename CT, bool GRAD>
__global__ void __launch_bounds__(256) k_lscan_chunk_scan(const LscanParams P) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= P.B * P.nc * P.M) return;
  const int64_t m = i % P.M, cj = (i / P.M) % P.nc, b = i / (P.M * P.nc);
  Chain<CT> ch{P, b, m};
  const int p0 = (int)cj * P.chunk;
  const int p1 = p0 + P.chunk < (int)P.L ? p0 + P.chunk : (int)P.L;
  CT h = ((const CT *)P.ws)[2 * P.B * P.nc * P.M + i], prod = 1;
  chunk_walk<CT, false, GRAD>(P, ch, p0, p1, h, prod);
}

// Row lanes per workgroup.  8 keep enough reads in flight from one workgroup per CU (256 workgroups of
// L 4096, forward + adjoint: 4 row lanes 165 + 349 us, 8 151 + 280, 16 164 + 338).  Two such
// workgroups fit a CU (registers; Hillis-Steele: LDS), so from 512 workgroups on, Hillis-Steele past
// it, 4 row lanes run in one round what 8 run in two (625 workgroups, hillis_steele, L 80 forward
// 16 -> 12 us), until 1,024 fill two rounds either way (L 2048: 326 us with 8, 340 with 4); short
// sequences keep 4, whose workgroups hide each other's latencies (forward + adjoint, 1,024
// workgroups, 8 -> 4: L 80 blelloch 46 -> 39, hillis_steele 45 -> 34; L 400 181 -> 178, 176 -> 169;
// L 1000 424 -> 443, 433 -> 429).  A sequence of at most 4, 2 or 1 row lanes' steps takes no more
// than these (sequential, 1,024 workgroups, 8 -> this: L 64 44 -> 26, L 16 39 -> 11).
template <typename CT, int ALGO, bool GRAD>
static hipError_t launch_walk(const LscanParams &all, hipStream_t s) {
  // A grid row holds fewer than 2^32 threads (more would wrap, unreported): wider scans take several.
  constexpr int64_t kMaxM = 1LL << 28;
  if (all.M > kMaxM) {
    for (int64_t m = 0; m < all.M; m += kMaxM) {
      LscanParams P = all;
      P.M = std::min(all.M - m, kMaxM);
      for (KView *v : {&P.a, &P.b, &P.h, &P.hf, &P.da}) v->p = v->p ? (CT *)v->p + m * v->s2 : nullptr;
      for (KView *v : {&P.h0, &P.h0f, &P.dh0}) v->p = v->p ? (CT *)v->p + m * v->s1 : nullptr;
      const hipError_t e = launch_walk<CT, ALGO, GRAD>(P, s);
      if (e != hipSuccess) return e;
    }
    return hipSuccess;
  }
  const LscanParams &P = all;
  const dim3 tiles((unsigned)((P.M + kScanMC - 1) / kScanMC), (unsigned)P.B);
  const int64_t g = lscan_groups(P.B, P.M);
  constexpr int R = scan_rows(ALGO);
  const bool four = g >= (ALGO == kHs ? 513 : 512) && (P.L <= 512 || g < 1024);
#define WALK(RL) hipLaunchKernelGGL((k_lscan_walk<CT, ALGO, RL, GRAD>), tiles, dim3(RL * kScanMC), 0, s, P)
  if (P.L <= R) WALK(1);
  else if (P.L <= 2 * R) WALK(2);
  else if (P.L <= 4 * R || four) WALK(4);
  else WALK(8);
#undef WALK
  return hipGetLastError();
}

// The one-wavefront kernel's conditions: unit stride along m, 16-byte aligned rows, M a multiple of
// 64.  It is taken where a workgroup's barriers cost more than its row lanes hide.  Forward, us,
// walk -> this: 16 workgroups, L 16 4.1 -> 3.0, L 48 5.0 -> 4.1, L 64 4.5 -> 5.1, L 80 6.4 -> 5.6,
// L 100 6.2 -> 6.8; 512 workgroups of L 2048 161 -> 154, 1,024 326 -> 308, 256 75 -> 94; 2,048 of
// L 80 24 -> 21, of L 400 139 -> 131, of L 1000 319 -> 325.
static bool seqt_ok(const LscanParams &P) {
  auto ok = [](const KView &v) {
    return v.s2 == 1 && v.s1 % 4 == 0 && v.s0 % 4 == 0 && ((uintptr_t)v.p % 16) == 0;
  };
  const int64_t g = lscan_groups(P.B, P.M);
  return P.M % kScanMC == 0 && ok(P.a) && ok(P.b) && ok(P.h) && 
         (P.L <= 48 || (P.L > 64 && P.L <= 96) || (g >= 512 && (g <= 1536 || P.L <= 512)));
}

template <typename CT, bool GRAD>
static hipError_t launch_lscan_t(const LscanParams &P, int algo, hipStream_t s) {
  switch (algo) {
    case kSeq:
      if constexpr (!GRAD && sizeof(CT) == 4) {
        if (!P.shift && seqt_ok(P)) {
          hipLaunchKernelGGL(k_lscan_seqt, dim3((unsigned)(P.M / kScanMC), (unsigned)P.B), dim3(kWave), 0, s, P);
          return hipGetLastError();
        }
      }
      return launch_walk<CT, kSeq, GRAD>(P, s);
    case kHs: return launch_walk<CT, kHs, GRAD>(P, s);
    case kBl: return launch_walk<CT, kBl, GRAD>(P, s);
  }
  // In one pass (each input read once) where its workgroups fill enough of the GPU, in three launches (a
  // and b read twice, every chunk in parallel) below.  Forward, forward + adjoint in us, one pass
  // against three launches, L 4096 float32: 192 workgroups 133, 328 against 208, 476; 160 127, 315
  // against 177, 398; 128 123, 306 against 141, 311; 96 122, 301 against 89, 231; L 16384, 64: 473,
  // 1174 against 300, 724.
  if (lscan_one_pass(P.B, P.M)) return launch_walk<CT, kChunk, GRAD>(P, s);
  const int64_t n = P.B * P.nc * P.M, chains = P.B * P.M;
  hipLaunchKernelGGL((k_lscan_chunk_reduce<CT>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, P);
  hipLaunchKernelGGL((k_lscan_chunk_carry<CT>), dim3((unsigned)((chains + 255) / 256)), dim3(256), 0, s, P);
  hipLaunchKernelGGL((k_lscan_chunk_scan<CT, GRAD>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, P);
  return hipGetLastError();
}

hipError_t launch_lscan(const LscanParams &P, int algo, int dtype, hipStream_t s) {
  if (P.hf.p) return dtype == 3 ? launch_lscan_t<double, true>(P, algo, s) : launch_lscan_t<float, true>(P, algo, s);
  return dtype == 3 ? launch_lscan_t<double, false>(P, algo, s) : launch_lscan_t<float, false>(P, algo, s);
}

}  // namespace ssm
