// The composed selective scan's kernels for the chunked algorithm with time segments (a translation unit
// of their own, beside the others in the build).
#include "ssm_cscan.hpp"

namespace ssm {
template hipError_t launch_csc_algo<kChunk, true>(const CscParams &, int, int, int, bool, hipStream_t);
}  // namespace ssm
