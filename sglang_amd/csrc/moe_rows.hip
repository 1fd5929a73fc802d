// Row-scaled fused-MoE grouped GEMMs (per-channel FP8 and INT8 experts, per-tensor FP8 experts) on the streaming and tile
// kernels of the block-scaled path.
//
// They used to run the register-staged generic kernel (gemm_core.h): 64 experts of 4096 x 1536, top-6, 250 tokens (1.2 GB
// of weights) took 186 + 114 us in its two GEMMs, 4.0 TB/s.
#include "moe_dispatch.h"

namespace sglamd {

// Whole K blocks and 32-bit buffer offsets; everything else stays with the generic kernel.
bool moe_rows_ok(const GemmArgs& g) {
  return (g.K % 128) == 0 && (g.K >> 7) <= GEMM8_BIG_MAX_KB && (int64_t)(g.num_valid / g.top_k) * g.lda < 0x7ffffff0ll &&
         (int64_t)g.N * g.ldb < 0x7ffffff0ll && gemm8_skinny_ok(g, g.num_valid / g.top_k);
}

int moe_rows_gemm(int mode, const GemmArgs& g, int out_dtype, int block_m, hipStream_t st) {
  SGLAMD_REQUIRE(out_dtype == SGLAMD_BF16 || out_dtype == SGLAMD_F16, SGLAMD_EINVAL,
                 "fused_moe_gemm: out_dtype must be Half or BFloat16");
  const DeviceScope scope;
  const bool bf16 = out_dtype == SGLAMD_BF16;
  if (mode == GEMM_ROW_INT8)
    return bf16 ? dispatch_moe_gemm<GEMM_ROW_INT8, BF16>(g, block_m, st)
                : dispatch_moe_gemm<GEMM_ROW_INT8, F16>(g, block_m, st);
  return bf16 ? dispatch_moe_gemm<GEMM_ROW_FP8, BF16>(g, block_m, st)
              : dispatch_moe_gemm<GEMM_ROW_FP8, F16>(g, block_m, st);
}

}  // namespace sglamd
