// The composed selective scan's kernels for one algorithm (a translation unit of their own: the
// build compiles the four side by side).
#include "ssm_cscan.hpp"

namespace ssm {
template hipError_t launch_csc_algo<kBl, false>(const CscParams &, int, int, int, bool, hipStream_t);
}  // namespace ssm
