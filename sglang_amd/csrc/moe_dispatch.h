// Which kernel a fused-MoE grouped GEMM over sorted blocks runs, by block height: shared by the block-scaled modes
// (moe.hip) and the row-scaled ones (moe_rows.hip).
#pragma once
#include <algorithm>
#include "gemm_big.h"
#include "gemm_big_moe_persist.h"
#include "gemm_moe_stream.h"
#include "gemm_skinny.h"

namespace sglamd {

// tuning knob: SGLAMD_MOE_PERSIST=0 runs the tall sorted blocks one tile per workgroup instead of the persistent walk
static inline bool moe_persist_enabled() {
  static const int v = getenv("SGLAMD_MOE_PERSIST") ? atoi(getenv("SGLAMD_MOE_PERSIST")) : 1;
  return v != 0;
}

// tuning knob: SGLAMD_MOE_PERSIST128=0 keeps the 128-slot sorted blocks with one tile per workgroup
static inline bool moe_persist128_enabled() {
  static const int v = getenv("SGLAMD_MOE_PERSIST128") ? atoi(getenv("SGLAMD_MOE_PERSIST128")) : 1;
  return v != 0 && moe_persist_enabled();
}

// tuning knob: SGLAMD_MOE_STREAM=0 keeps the weight-streaming tile kernel out
static inline bool moe_stream_enabled() {
  static const int v = getenv("SGLAMD_MOE_STREAM") ? atoi(getenv("SGLAMD_MOE_STREAM")) : 1;
  return v != 0;
}
// Whether the weight-streaming tile kernel takes a launch: weights that come from HBM.  A layer of less than some 96 MB of
// weights may find them in the 256 MB Infinity Cache from one call to the next; there the one-tile kernel, which starts a
// tile sooner, is ahead (three layers used in turn, 12 rows per expert, one-tile kernel over this one: 8 experts of
// 3072 x 1024 0.80, 16 of 1536 x 640 0.92; 64 of 1024 x 512, 101 MB, 1.13, 32 of 2048 x 768, 151 MB, 1.06).  With weights that have left the cache this one
// is ahead on all of them (1.0-1.12x).
constexpr int64_t MOE_STREAM_MIN_BYTES = 96000000;
// The same for a grouped GEMM called on its own, which knows its list of sorted blocks but not how many experts there are.  A
// list has room for the pairs and for block_m - 1 slots of padding per expert, so what is left beside the pairs says how
// many experts it was made for; the blocks themselves do not (8192 pairs of 8 experts are 136 blocks of 64).
static inline bool moe_list_streams(int64_t num_valid, int64_t max_blocks, int block_m, int64_t N, int64_t ldb) {
  const int64_t experts = std::min(num_valid, (max_blocks * block_m - num_valid) / (block_m - 1));
  return experts * N * ldb >= MOE_STREAM_MIN_BYTES * 2 / 3;
}
template <int BM>
static inline bool moe_stream_takes(const GemmArgs& g, bool block) {
  if (g.streams < 0 || !moe_stream_enabled() || !gemm8_moe_stream_ok<BM>(g, block)) return false;
  return g.streams > 0 || moe_list_streams(g.num_valid, g.max_blocks_m, BM, g.N, g.ldb);
}

// The persistent walk hands out tiles by position, not by arrival.  A sorted block that is an expert's second one
// finds the weights its first block has just streamed in L2 and finishes in half the time, and a fixed walk cannot
// balance that the way the dispatch order of a one-tile-per-workgroup launch does; until the tiles went to XCDs in
// contiguous ranges the walk therefore lost 5 % where half of the experts own one block and half two (6144 tokens
// on the DeepSeek-V3 layer) and was only used where every expert owns the same number.  With an expert's blocks
// meeting in one L2 it is level or ahead at every token count measured (3072 ... 12288: 0 ... -5.5 %), so it runs
// wherever there are more tiles than CUs.
template <int MODE, typename OT>
static int dispatch_moe_gemm(const GemmArgs& g, int block_m, hipStream_t st) {
  // number of sorted blocks that will actually run is data dependent; every valid slot could own one
  const int64_t expect = g.num_valid < g.max_blocks_m ? g.num_valid : g.max_blocks_m;
  const bool streaming_ok = gemm8_skinny_ok(g, g.num_valid / g.top_k);
  switch (block_m) {
    case 16:
      if (streaming_ok) return gemm8_skinny_launch<1, MODE, OT, true>(g, st, expect);
      return gemm8_launch<16, 128, 1, 2, MODE, OT, true>(g, st);  // operands of 2 GiB and more
    case 32:
      if (streaming_ok) return gemm8_skinny_launch<2, MODE, OT, true>(g, st, expect);
      return gemm8_launch<32, 128, 1, 2, MODE, OT, true>(g, st);
    case 64:
      if (moe_stream_takes<64>(g, gemm_is_block(MODE)))
        return gemm8_moe_stream_launch<MODE, OT, 64>(g, st);
      // the tile kernel with one 32-row tile per wave when its preconditions hold: the streaming kernel spends
      // four MFMA row groups per weight fragment and falls far behind it at this height
      if ((g.K % 128) == 0 && (g.K >> 7) <= GEMM8_BIG_MAX_KB && (int64_t)(g.num_valid / g.top_k) * g.lda < 0x7fffffffll &&
          (int64_t)g.N * g.ldb < 0x7fffffffll)
        // (the persistent walk with its two stages is 12 % behind this kernel's three at this height)
        return gemm8_big_moe_launch<MODE, OT, 1>(g, st);
      if (streaming_ok) return gemm8_skinny_launch<4, MODE, OT, true>(g, st, expect);
      return gemm8_launch<64, 128, 2, 2, MODE, OT, true>(g, st);
    case 128:
      if constexpr (!gemm_is_block(MODE)) {
        if (moe_stream_takes<128>(g, false)) return gemm8_moe_stream_launch<MODE, OT, 128>(g, st);
      }
      // 32x32x64-MFMA tile kernel when its preconditions hold (K % 128 == 0, operands below 2 GiB per matrix)
      if ((g.K % 128) == 0 && (g.K >> 7) <= GEMM8_BIG_MAX_KB && (int64_t)(g.num_valid / g.top_k) * g.lda < 0x7fffffffll &&
          (int64_t)g.N * g.ldb < 0x7fffffffll)
      {
        // more tiles than CUs: the persistent walk, as for the 192-slot blocks
        if constexpr (gemm_is_block(MODE)) {
          if (moe_persist128_enabled() && gemm8_moe_persist_ok(g) &&
              (int64_t)((g.N + 255) / 256) * g.max_blocks_m > device_cus())
            return gemm8_moe_persist_launch<MODE, OT, 2>(g, st);
        }
        return gemm8_big_moe_launch<MODE, OT>(g, st);
      }
      return gemm8_launch<128, 128, 2, 2, MODE, OT, true>(g, st);
    case 192:
      // one block per expert when an expert gets 129..192 rows: its weights are streamed once
      SGLAMD_REQUIRE((g.K % 128) == 0 && (g.K >> 7) <= GEMM8_BIG_MAX_KB && (int64_t)(g.num_valid / g.top_k) * g.lda < 0x7fffffffll &&
                         (int64_t)g.N * g.ldb < 0x7fffffffll,
                     SGLAMD_EINVAL, "fused_moe_gemm: block_m 192 needs K %% 128 == 0 and operands below 2 GiB");
      // more tiles than CUs: one workgroup per CU walks them and requests a tile's first blocks under the
      // epilogue of the tile before
      if constexpr (gemm_is_block(MODE)) {
        if (moe_persist_enabled() && gemm8_moe_persist_ok(g) &&
            (int64_t)((g.N + 255) / 256) * g.max_blocks_m > device_cus())
          return gemm8_moe_persist_launch<MODE, OT, 3>(g, st);
      }
      return gemm8_big_moe_launch<MODE, OT, 3>(g, st);
    default:
      return fail(SGLAMD_EINVAL, "fused_moe_gemm: block_m must be 16, 32, 64, 128 or 192 (got %d)", block_m);
  }
}

// The row-scaled grouped GEMMs (moe_rows.hip): per-token or per-tensor activation scales, per-channel or per-expert
// weight scales, optional bias; see GemmArgs for where their strides sit.
bool moe_rows_ok(const GemmArgs& g);
int moe_rows_gemm(int mode, const GemmArgs& g, int out_dtype, int block_m, hipStream_t st);

}  // namespace sglamd
