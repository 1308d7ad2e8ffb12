// The four scan algorithms on one time tile held in registers, shared by the linear scans
// (ssm_lscan.hip) and the composed selective scan (ssm_cscan.hip).
//
// A workgroup's wavefronts are the tile's row lanes: row lane tr holds R of the tile's RL * R steps
// for 64 neighbouring recurrences (one per lane), as the affine maps h <- a h + b.  tile_scan turns
// b into the states; what passes between the row lanes goes through LDS.
#pragma once

#include "ssm_device.hpp"
#include "ssm_wave.hpp"

namespace ssm {

enum { kSeq = 1, kHs = 2, kBl = 3, kChunk = 4 };  // algorithm ids of the C ABI

// A row lane's r-th step of the tile: R consecutive steps, or every RL-th (Hillis-Steele).
template <int ALGO, int RL, int R>
__device__ __forceinline__ int tile_step(int tr, int r) {
  return ALGO == kHs ? tr + RL * r : tr * R + r;
}

// What the row lanes exchange through LDS.  A call may start while another wavefront still reads
// the last values of the call before it: those are never in the half (or array) written first.
template <typename CT, int ALGO, int RL, int R> struct TileLds {  // sequential: the state handed over
  CT h[2][kWave];
};
template <typename CT, int RL, int R> struct TileLds<CT, kHs, RL, R> {
  CT A[2][RL * R][kWave], S[2][RL * R][kWave], last[kWave];
};
template <typename CT, int RL, int R> struct TileLds<CT, kBl, RL, R> {
  CT A[RL][kWave], S[RL][kWave], last[kWave];
};
template <typename CT, int RL, int R> struct TileLds<CT, kChunk, RL, R> {
  CT P[2][RL][kWave], E[2][RL][kWave];
};

struct NoEmit {
  __device__ __forceinline__ void operator()() const {}
};

// b[r] becomes the state after step r; carry, the state entering the tile, the state leaving it
// (the same bits in every row lane); hin the state entering the row lane's block (consecutive
// steps only).  a is overwritten by Hillis-Steele.  buf: parity of the double-buffered halves.
// emit() is called once b holds the states, ahead of what the row lanes still wait for (stores issued
// there overlap the last barrier: Blelloch, 128 workgroups of L 4096, forward 130 -> 121 us).
template <typename CT, int ALGO, int RL, int R, typename EMIT = NoEmit>
__device__ __forceinline__ void tile_scan(TileLds<CT, ALGO, RL, R> &X, CT (&a)[R], CT (&b)[R], CT &carry, CT &hin,
                                          int tr, int mi, int &buf, EMIT emit = EMIT{}) {
  if constexpr (ALGO == kSeq) {
    // The row lanes take turns: a handover and R dependent updates each.  (RL is even, or 1: the next
    // call's first turn writes the half that the last handover of this one is not in.)
    static_assert(RL == 1 || RL % 2 == 0, "row lanes");
#pragma unroll
    for (int q = 0; q < RL; ++q) {
      if (q == tr) {
        CT h = q == 0 ? carry : X.h[(q + 1) & 1][mi];
        hin = h;
#pragma unroll
        for (int r = 0; r < R; ++r) {
          h = fma(a[r], h, b[r]);
          b[r] = h;
        }
        X.h[q & 1][mi] = h;
      }
      lds_barrier();
    }
    carry = X.h[(RL - 1) & 1][mi];
    emit();
  } else if constexpr (ALGO == kHs) {
    // At offset o every step k >= o composes with step k - o of the previous pass.  The
    // offsets below RL pair different row lanes (step k - o is in row lane tr - o, or one
    // register lower in row lane tr - o + RL), the others registers of one lane.
    if (tr == 0) b[0] = fma(a[0], carry, b[0]);  // fold the incoming state into the first element
#pragma unroll
    for (int o = 1; o < RL; o *= 2) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        X.A[buf][tr + RL * r][mi] = a[r];
        X.S[buf][tr + RL * r][mi] = b[r];
      }
      lds_barrier();
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int k = tr + RL * r;
        if (k >= o) {
          b[r] = fma(a[r], X.S[buf][k - o][mi], b[r]);
          a[r] = a[r] * X.A[buf][k - o][mi];
        }
      }
      buf ^= 1;  // the next pass (or call) writes beside the steps still being read
    }
#pragma unroll
    for (int j = 1; j < R; j *= 2) {  // descending r reads the previous pass's r - j
#pragma unroll
      for (int r = R - 1; r >= j; --r) {
        b[r] = fma(a[r], b[r - j], b[r]);
        a[r] = a[r] * a[r - j];
      }
    }
    if (tr == RL - 1) X.last[mi] = b[R - 1];
    emit();
    lds_barrier();
    carry = X.last[mi];
  } else if constexpr (ALGO == kBl) {
    // Tree levels of span 2..R are register operations of one lane; the levels above combine
    // the block roots, which every lane of a column reads from LDS and sweeps itself (the
    // same combines in every lane, so the same bits).
    CT A[R], S[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      A[r] = a[r];
      S[r] = b[r];
    }
#pragma unroll
    for (int sp = 2; sp <= R; sp *= 2) {  // up-sweep: right <- right o left at nodes (j + 1) sp - 1
#pragma unroll
      for (int k = sp - 1; k < R; k += sp) {
        const int l = k - sp / 2;
        S[k] = fma(A[k], S[l], S[k]);
        A[k] = A[k] * A[l];
      }
    }
    X.A[tr][mi] = A[R - 1];
    X.S[tr][mi] = S[R - 1];
    lds_barrier();
    CT rA[RL], rS[RL];
#pragma unroll
    for (int q = 0; q < RL; ++q) {
      rA[q] = X.A[q][mi];
      rS[q] = X.S[q][mi];
    }
#pragma unroll
    for (int sp = 2; sp <= RL; sp *= 2) {
#pragma unroll
      for (int k = sp - 1; k < RL; k += sp) {
        const int l = k - sp / 2;
        rS[k] = fma(rA[k], rS[l], rS[k]);
        rA[k] = rA[k] * rA[l];
      }
    }
    // the root set to the identity, then the down-sweep (left <- right; right <- left_old o
    // right): each root becomes the composition of the blocks before it
    rA[RL - 1] = 1;
    rS[RL - 1] = 0;
#pragma unroll
    for (int sp = RL; sp >= 2; sp /= 2) {
#pragma unroll
      for (int k = sp - 1; k < RL; k += sp) {
        const int l = k - sp / 2;
        const CT tA = rA[l], tS = rS[l];
        rA[l] = rA[k];
        rS[l] = rS[k];
        rS[k] = fma(rS[k], tA, tS);
        rA[k] = rA[k] * tA;
      }
    }
#pragma unroll
    for (int q = 0; q < RL; ++q) {  // this row lane's root
      if (q == tr) {
        A[R - 1] = rA[q];
        S[R - 1] = rS[q];
      }
    }
#pragma unroll
    for (int sp = R; sp >= 2; sp /= 2) {
#pragma unroll
      for (int k = sp - 1; k < R; k += sp) {
        const int l = k - sp / 2;
        const CT tA = A[l], tS = S[l];
        A[l] = A[k];
        S[l] = S[k];
        S[k] = fma(S[k], tA, tS);
        A[k] = A[k] * tA;
      }
    }
    // exclusive prefixes: the state entering step k is A_k h_in + S_k
    hin = fma(A[0], carry, S[0]);
#pragma unroll
    for (int r = 0; r < R; ++r) b[r] = fma(a[r], fma(A[r], carry, S[r]), b[r]);
    if (tr == RL - 1) X.last[mi] = b[R - 1];
    emit();
    lds_barrier();
    carry = X.last[mi];
  } else {
    CT pr = a[0], e = b[0];
#pragma unroll
    for (int r = 1; r < R; ++r) {
      e = fma(a[r], e, b[r]);
      pr *= a[r];
    }
    X.P[buf][tr][mi] = pr;
    X.E[buf][tr][mi] = e;
    lds_barrier();
    CT h = carry;
#pragma unroll
    for (int q = 0; q < RL; ++q) {  // the same folds in every lane, so the same bits
      if (q == tr) h = carry;       // the state entering this row lane's chunk
      carry = fma(X.P[buf][q][mi], carry, X.E[buf][q][mi]);
    }
    hin = h;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      h = fma(a[r], h, b[r]);
      b[r] = h;
    }
    emit();
    buf ^= 1;  // the next call's summaries go beside the ones still being read
  }
}

}  // namespace ssm
