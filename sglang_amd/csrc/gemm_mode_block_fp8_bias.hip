// Every dense GEMM kernel in the GEMM_BLOCK_FP8 scaling mode with a bias added to the output (see gemm_dispatch.h).
#include "gemm_dispatch.h"

namespace sglamd {
template int dispatch_out_biased<GEMM_BLOCK_FP8>(const GemmArgs&, int, hipStream_t, void*, int64_t);
template int dispatch_quantising<GEMM_BLOCK_FP8, true>(const GemmArgs&, int, hipStream_t, bool);
}  // namespace sglamd
