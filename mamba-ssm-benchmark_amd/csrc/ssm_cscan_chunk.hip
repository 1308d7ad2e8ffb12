// The composed selective scan: the chunked algorithm's kernels, the final sums of the backward's
// partials and the dispatch over the algorithms.
#include <algorithm>

#include "ssm_cscan.hpp"

namespace ssm {

template hipError_t launch_csc_algo<kChunk, false>(const CscParams &, int, int, int, bool, hipStream_t);
extern template hipError_t launch_csc_algo<kSeq, false>(const CscParams &, int, int, int, bool, hipStream_t);
extern template hipError_t launch_csc_algo<kHs, false>(const CscParams &, int, int, int, bool, hipStream_t);
extern template hipError_t launch_csc_algo<kBl, false>(const CscParams &, int, int, int, bool, hipStream_t);
extern template hipError_t launch_csc_algo<kChunk, true>(const CscParams &, int, int, int, bool, hipStream_t);

// dBm, dCm: the channel tiles' partials of each (b, t, n); dA: the batch rows' (and segments').  Float64 sums in
// index order, the reads of 16 terms issued together.
template <typename CT>
__global__ void __launch_bounds__(kThreads) k_csc_fin(const CscParams p, int np) {
  const int64_t row = 2 * np, nBC = p.B * p.L * row, nA = p.D * p.N;
  for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < nBC + nA; i += (int64_t)gridDim.x * kThreads) {
    if (i < nBC) {
      const int64_t n = i % np, q = (i / np) % 2, t = (i / row) % p.L, b = i / (row * p.L);
      if (n >= p.N) continue;
      const CT *src = (const CT *)p.ws_bc + (b * p.ntiles * p.L + t) * row + q * np + n;
      const CT s = (CT)ordered_sum<16, CT, double>(src, p.L * row, p.ntiles);
      const KView &o = q ? p.dC : p.dB;
      vstore<CT>(o, b * o.s0 + t * o.s1 + n * o.s2, s);
    } else {
      const int64_t j = i - nBC, n = j % p.N, d = j / p.N;
      const double s = ordered_sum<16>((const double *)p.ws_dA + j, nA, p.B * p.nseg);
      vstore<CT>(p.dA, d * p.dA.s0 + n * p.dA.s1, (CT)s);
    }
  }
}

hipError_t launch_csc(const CscParams &p, int algo, int dtype, int method, int np, bool bwd, hipStream_t s) {
  hipError_t e;
  switch (algo) {
    case kSeq: e = launch_csc_algo<kSeq, false>(p, dtype, method, np, bwd, s); break;
    case kHs: e = launch_csc_algo<kHs, false>(p, dtype, method, np, bwd, s); break;
    case kBl: e = launch_csc_algo<kBl, false>(p, dtype, method, np, bwd, s); break;
    default:
      e = p.nseg > 1 ? launch_csc_algo<kChunk, true>(p, dtype, method, np, bwd, s)
                     : launch_csc_algo<kChunk, false>(p, dtype, method, np, bwd, s);
  }
  if (e != hipSuccess || !bwd) return e;
  const int64_t n = p.B * p.L * 2 * np + p.D * p.N;
  constexpr int64_t kMaxBlocks = 1 << 23;  // a launch holds fewer than 2^32 threads: 2^31, each striding on
  const dim3 grid((unsigned)std::min((n + kThreads - 1) / kThreads, kMaxBlocks));
  if (dtype == 3) hipLaunchKernelGGL((k_csc_fin<double>), grid, dim3(kThreads), 0, s, p, np);
  else hipLaunchKernelGGL((k_csc_fin<float>), grid, dim3(kThreads), 0, s, p, np);
  return hipGetLastError();
}

}  // namespace ssm
