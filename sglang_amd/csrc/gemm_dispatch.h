// Which kernel a dense 8-bit GEMM call runs, by shape: shared by the per-mode translation units (gemm_mode_*.hip,
// one explicit instantiation of dispatch_out each, so that they compile in parallel) and the entry points (gemm.hip).
#pragma once
#include <stdlib.h>

#include "gemm_big.h"
#include "gemm_big_persist.h"
#include "gemm_skinny.h"
#include "gemm_strip.h"

namespace sglamd {

// Width of the large-M tile in 64-column wave tiles (4 -> 256x256, 2 -> 256x128); tuning knob.
static int big_wgn() {
  static const int v = getenv("SGLAMD_BIG_WGN") ? atoi(getenv("SGLAMD_BIG_WGN")) : 4;
  return v;
}

// Rows from which the tile kernel takes over from the streaming kernel; tuning knob.
static int tile_min_m() {
  static const int v = getenv("SGLAMD_TILE_MIN_M") ? atoi(getenv("SGLAMD_TILE_MIN_M")) : 17;
  return v;
}

// 33 to 64 rows: the tile kernel (64-row tile, K split over the chip) or the streaming kernel, where dense_choice below has nothing
// faster?  Up to 32 rows the streaming kernel is the faster of these two on every weight measured (past 100 MB strips are: dense_choice; DeepSeek-V3 gate_up / down / q_b / o_proj at 17 rows:
// 54.5 / 26.1 / 12.1 / 22.8 us against 60.0 / 31.7 / 16.9 / 28.8 in 64-row tiles; at 32 rows 63.9 / 30.4 / 13.9 / 25.6
// against 61.6 / 32.6 / 17.3 / 30.0; Llama-3-70B o / gate_up / down at 24 rows 15.0 / 86.6 / 43.2 against 19.3 / 104.5 /
// 50.6).  Its four-tile form for 33..64 rows re-reads the activations too often for large weights (gate_up at 48
// rows: 83.9 us against 63.5), but a launch of the tile kernel costs more (a second kernel when K is split) and it
// needs about a hundred workgroups to hide its per-block latency, so small weights stay with the streaming kernel.
// Rows of a ragged K start anywhere in a 128-byte line, which the tile kernel's loads (8 rows each) pay for more than
// the streaming kernel's: there it takes 80 column tiles, or 48 of a long K (8192 x 4112 at 40 rows 20 us in tiles, 17
// streamed; 12288 20 against 24, 20480 25 against 35, 28672 29 against 46).
static bool small_m_uses_tile(int64_t M, int64_t N, int64_t K) {
  if (M < tile_min_m() || M <= 32) return false;
  const int64_t tiles = (N + 255) / 256;
  if (K & 127) return tiles >= 80 || (tiles >= 48 && K >= 4096);
  const int slices = gemm8_big_slices(tiles, N, K);
  if (tiles * slices >= 96) return true;
  return (slices == 1 && tiles >= 32) || K >= 6144;
}

// The wide streaming form for 33..64 rows (tuning knob: 0 switches it off).
static bool wide_streaming() {
  static const int v = getenv("SGLAMD_WIDE") ? atoi(getenv("SGLAMD_WIDE")) : 1;
  return v != 0;
}

// Workgroups of the persistent large-tile kernel: one per CU of the current device (0: kernel switched off).
static int persist_workgroups() {
  static const int off = getenv("SGLAMD_BIG_PERSIST") ? atoi(getenv("SGLAMD_BIG_PERSIST")) == 0 : 0;
  return off ? 0 : device_cus();
}

// Which kernel the last dense GEMM call of this thread launched (SGLAMD_KERNEL_* of the header): lets a test
// assert that it exercises the kernel it was written for, whatever the launch heuristics choose.
extern thread_local int last_kernel, strip_last_shape;  // defined in gemm.hip
#define RAN(code) (last_kernel = (code))

// A launch of 256x256 tiles whose last round of one tile per CU is mostly empty is cut in two along N: the
// columns that fill whole rounds, and the rest as a launch of its own, which picks the tile height and K split that
// fill the chip with what is left.
// Returns the columns of the first part (a multiple of 256), or 0 to leave the launch whole.  Measured on the
// DeepSeek-V3 gate_up weight (N = 36864, K = 7168): M = 512 179 -> 147 us, M = 1024 303 -> 279 us, while at
// M = 2048 (four and a half rounds) the two launches cost more than the half round they save.
static int64_t column_split(int64_t M, int64_t N, int64_t K) {
  static const int off = getenv("SGLAMD_BIG_COLSPLIT") ? atoi(getenv("SGLAMD_BIG_COLSPLIT")) == 0 : 0;
  if (off || M <= 128 || (N & 255)) return 0;
  const int64_t cus = device_cus();
  const int64_t tiles_m = (M + 255) / 256, tiles_n = N / 256, tiles = tiles_m * tiles_n;
  const int64_t rounds = tiles / cus, tail = tiles % cus;
  if (rounds < 1 || rounds > 2 || tail == 0 || tail * 8 > cus * 3) return 0;
  const int64_t first = rounds * cus / tiles_m;  // column tiles that make up the whole rounds
  if (first < 1 || first >= tiles_n) return 0;
  return first * 256;
}

// 17 to 1024 rows: the tile kernels (or, up to 64 rows, what small_m_uses_tile says), the strip kernel, or the streaming kernel walking
// several row tiles?  Small weights are not worth a tile launch: it leaves most of the chip idle, or splits K and needs a second
// launch, where the streaming kernel's small tiles fill it (2048 x 2048 at 128 rows, quantiser included, 15.2 -> 8.7 us, 1024 x 7168
// 17.6 -> 12.3, 512 x 512 at 320 rows 8.7 -> 6.5), until reading the weights once per row tile costs more (4096 x 4096 at 150 rows
// 20 -> 23).  The strip kernel takes over from weights of about 25 MB (28672 x 4096 at 64 / 128 rows 35 / 40 -> 27 / 33 us, 7168 x 16384
// 38 / 48 -> 33 / 41).  The line between them is drawn by each form's time from a fitted model.  Over 2335 points (186 weights from
// HBM, three scaling modes) and 949 (three weights in turn, up to 85 MB, so from the Infinity Cache): 1.13x in the mean of
// either, 0.98 of the fastest form's, the worst point 0.93x, eight below 0.97.
// Row tiles of 16 rows instead of 32, at 17 to 64 rows: a shorter chain per wave, at twice the reads, so only while the weights are
// a few MB (704 x 4736 at 24 rows 10.6 -> 9.9 us, 1152 x 7040 16.0 -> 14.2; 4096 x 4096 11.6 -> 12.4).
// Strips at 17 to 32 rows: weights of 100 MB and more in tiles of 96 to 160 rows that fill 0.85 of their rounds (36864 x 7168 at 24 / 32
// rows 49 / 51 -> 45 / 46 us, 40000 x 4096 36 / 37 -> 31, 57344 x 8192 79 / 81 -> 76 / 77; 42 points 1.05x in the mean, the worst 0.95x).
// Narrower tiles (20000 x 8192 in tiles of 80: 33.5 -> 39), K slices (10240 x 16384 33 -> 37) and smaller weights (24576 x 1536 from HBM 13
// -> 14) stay with the streaming kernel.
// A ragged K: rows start anywhere in a 128-byte line, and every form pays for it, by the factors below (the mean over 720 points to
// their models).  512 x 1424 at 96 rows 13.6 -> 7.3 us, 23800 x 5984 at 80 rows 62 -> 45; beyond 128 rows only weights up to 2 MB
// (512 x 1424 at 200 rows 13.7 -> 7.4, 848 x 1904 15.4 -> 10.1; 680 x 4768 at 320 rows 19.7 against 18.9).
struct DenseChoice {
  int row_tile = 0;  // streaming kernel in row tiles of this many rows
  StripPlan strip;   // strip.rows > 0: strip kernel
};
static DenseChoice dense_choice(int64_t M, int64_t N, int64_t K) {
  DenseChoice best;
  const bool ragged = (K & 127) != 0;
  if (M <= 16 || M > 1024 || (ragged && M > 128 && N * K > 2000000)) return best;
  // the models are a few microseconds of host time: a thread remembers its last shapes (see skinny_plan)
  struct Known {
    int64_t M, N, K, cus;
    DenseChoice choice;
  };
  static thread_local Known known[32] = {};
  const int64_t cus = device_cus();
  Known& slot = known[((uint32_t)M * 31u + (uint32_t)(N >> 3) * 7u + (uint32_t)(K >> 7)) & 31u];
  if (slot.M == M && slot.N == N && slot.K == K && slot.cus == cus) return slot.choice;

  const double common = 5.0 + 0.7e-6 * M * K;  // launch and quantiser
  bool fills[3];
  double small[3] = {M <= 64 ? skinny_row_tiles_us<1>(M, N, K, &fills[0]) * (ragged ? 1.25 : 1.0) : 1e30,
                     skinny_row_tiles_us<2>(M, N, K, &fills[1]) * (ragged ? 1.25 : 1.0),
                     M > 32 ? skinny_row_tiles_us<4>(M, N, K, &fills[2]) * (ragged ? 1.15 : 1.0) : 1e30};
  const bool streamed = M <= 64 && !small_m_uses_tile(M, N, K);  // without this choice: the streaming kernel's 32- or 64-row tile
  int small_rows = 32;
  if (M <= 64 && (streamed || fills[0]) && small[0] * 1.02 + 0.02 * common < small[1] && N * K <= 10000000)
    small_rows = 16, small[1] = small[0], fills[1] = true;
  if (M <= 32) {  // the streaming kernel, one tile of 32 rows or two of 16, or strips of weights too large for the caches
    if (small_rows == 16) best.row_tile = 16;
    const StripPlan plan = N * K >= 100000000 ? strip_plan(M, N, K) : StripPlan();
    const int64_t tiles = plan.rows ? ceil_div(N, plan.rows) : 0;
    if (plan.rows >= 96 && plan.slices == 1 && tiles * 20 >= ceil_div(tiles, cus) * cus * 17) best.strip = plan;
    slot = Known{M, N, K, cus, best};
    return best;
  }
  double least;
  bool row_tiles = true;
  if (streamed) {
    least = common + small[2];
  } else {
    const int nkb = (int)((K + 127) >> 7);
    const bool persistent = !ragged && !(nkb & 1) && nkb >= 4 && nkb <= GEMM8_PERSIST_USE_MAX_KB;
    const BigConfig cfg = gemm8_big_config(M, N, K, persistent);
    const int64_t cols = ceil_div(N, 256) * cfg.slices, rounds = ceil_div(ceil_div(M, cfg.bm) * cols, cus);
    // a K block of a tile, or of the weights that the column tiles in flight read (6.7 TB/s from the Infinity Cache, 5.2 else)
    const double block = std::max(cfg.bm == 64 ? 0.52 : cfg.bm == 128 ? 1.04 : cfg.bm == 192 ? 1.45 : 1.85, (N * K > 85000000 ? 0.0063 : 0.0049) * std::min(cols, cus));
    double us = rounds * ((double)nkb / cfg.slices * block + 2.2);
    row_tiles = M > 64 || cfg.slices > 1;  // up to 64 rows the model is not fine enough to tell them from one launch of 64-row tiles
    if (cfg.slices > 1) us += 3.2 + 1.86e-6 * cfg.slices * M * N;
    least = common + us * (ragged ? 1.15 : 1.0);
  }
  for (int f = 1; f < 3 && row_tiles; f++) {
    if (!fills[f]) continue;
    const double us = (common + small[f]) * (streamed && f == 2 ? 1.0 : ragged && M > 128 ? 1.25 : 1.12);
    if (us < least) least = us, best.row_tile = f == 2 ? 64 : small_rows;
  }
  if (M <= STRIP_MAX_ROWS) {
    const StripPlan plan = strip_plan(M, N, K);
    // (on large weights with a K of some length the tile kernel is slower than its model; not with K split, or half of the CUs, at more than 96 rows on
    // weights that come from the Infinity Cache: 8192 x 8192 at 114 / 128 rows 25.4 / 26.0 us, 26.6 / 27.6 in strips,
    // 12288 x 4096 at 128 rows 22.4 and 24.0)
    const double margin = N * K < 30000000 || K < 2560 ? 1.1 : M > 96 && N * K < 75000000 && (plan.slices > 1 || ceil_div(N, plan.rows) * 2 < cus) ? 1.0 : 0.93;
    if ((common + plan.us * (ragged ? 1.12 : 1.0)) * margin < least) best.row_tile = 0, best.strip = plan;
  }
  slot = Known{M, N, K, cus, best};
  return best;
}

// The same for a test (sglamd_dense_plan): operands without gaps, 16-byte aligned scratch of the size that
// sglamd_gemm_workspace_bytes reports.
static inline int dense_plan(bool block, int64_t M, int64_t N, int64_t K, int32_t* plan) {
  const DenseChoice choice = block && (K & 127) ? DenseChoice() : dense_choice(M, N, K);
  plan[0] = plan[1] = plan[2] = plan[3] = 0;
  if (choice.row_tile) {
    plan[0] = choice.row_tile;
    return SGLAMD_PLAN_ROW_TILES;
  }
  if (choice.strip.rows && (!block || strip_tables_hold(M, N, K, choice.strip))) {
    plan[0] = (int32_t)((M + 31) / 32 * 32), plan[1] = choice.strip.rows, plan[2] = choice.strip.slices, plan[3] = strip_depth(M, choice.strip.rows);
    return SGLAMD_PLAN_STRIPS;
  }
  if (M <= 64 && !small_m_uses_tile(M, N, K)) return SGLAMD_PLAN_STREAMING;
  const int64_t nkb = K >> 7;
  const BigConfig cfg = gemm8_big_config(M, N, K, block && !(nkb & 1) && nkb >= 4 && nkb <= GEMM8_PERSIST_USE_MAX_KB);
  plan[0] = cfg.bm, plan[1] = 256, plan[2] = cfg.slices;
  return SGLAMD_PLAN_TILES;
}

// The row modes' tile kernel also takes a K that is not a multiple of 128, from 512 up: 8192 x 4112 at 100 / 300 / 1000 rows
// 43 / 45 / 60 -> 21 / 32 / 46 us (4096: 20 / 23 / 39), 28672 x 4112 at 2048 rows 407 -> 281.  Shorter sums are a launch of
// 12 to 17 us either way and stay with the generic kernel.
template <int MODE, typename OT>
static int dispatch_dense(const GemmArgs& g, hipStream_t st, void* workspace, int64_t workspace_bytes,
                          bool may_split = true) {
  RAN(SGLAMD_KERNEL_STREAMING);
  const bool big = gemm8_big_ok(g, !gemm_is_block(MODE) && g.K >= 512);
  const int wgs = gemm_is_block(MODE) ? persist_workgroups() : 0;
  const int nkb = g.K >> 7;
  const bool persistent = wgs > 0 && (wgs & 7) == 0 && !(nkb & 1) && nkb >= 4 && nkb <= GEMM8_PERSIST_USE_MAX_KB;
  const int tiles_256 = persistent ? (MODE == GEMM_BLOCK_FP8 && g.scales_pow2 ? 2 : 1) : 0;
  strip_last_shape = skinny_last_shape = 0;
  if (big && may_split && g.M > 16) {
    const DenseChoice choice = dense_choice(g.M, g.N, g.K);
    const StripPlan& plan = choice.strip;
    if (choice.row_tile && gemm8_skinny_ok(g, g.M)) {
      if (choice.row_tile == 64) return gemm8_skinny_launch<4, MODE, OT, false>(g, st, ceil_div(g.M, 64));
      if (choice.row_tile == 16) return gemm8_skinny_launch<1, MODE, OT, false>(g, st, ceil_div(g.M, 16));
      return gemm8_skinny_launch<2, MODE, OT, false>(g, st, ceil_div(g.M, 32));
    }
    if (plan.rows && strip_ok<MODE>(g, plan) &&
        (plan.slices == 1 || (workspace && ((uintptr_t)workspace & 15) == 0 && (int64_t)plan.slices * g.M * g.N * 4 <= workspace_bytes))) {
      RAN(SGLAMD_KERNEL_STRIP);
      strip_last_shape = ((g.M + 31) / 32 << 24) | (plan.slices << 16) | plan.rows;
      return gemm8_strip_launch<MODE, OT>(g, plan, st, workspace);
    }
  }
  if (big && may_split && g.M > 64) {
    const BigConfig whole = gemm8_big_config(g.M, g.N, g.K, tiles_256);
    const int64_t n1 = whole.bm == 256 && whole.slices == 1 ? column_split(g.M, g.N, g.K) : 0;
    if (n1 > 0) {
      typedef typename OT::storage OS;
      GemmArgs head = g, rest = g;
      head.N = (int)n1;
      rest.N = g.N - (int)n1;
      rest.B = g.B + n1 * g.ldb;
      rest.C = (OS*)g.C + n1;
      rest.sb = gemm_is_block(MODE) ? g.sb + (n1 >> 7) * g.sb_sn : g.sb + n1;
      if (g.bias) rest.bias = (const OS*)g.bias + n1;
      int rc = dispatch_dense<MODE, OT>(head, st, workspace, workspace_bytes, false);
      if (rc) return rc;
      const int ran = last_kernel;
      rc = dispatch_dense<MODE, OT>(rest, st, workspace, workspace_bytes, false);
      RAN(ran);  // the kernel that did most of the work
      return rc;
    }
  }
  if (gemm8_skinny_ok(g, g.M)) {
    if (g.M > 32 && g.M <= 64 && wide_streaming() && gemm8_skinny_wide<MODE, OT>(g, st, false) > 0) {
      RAN(SGLAMD_KERNEL_STREAMING_WIDE);
      return gemm8_skinny_wide<MODE, OT>(g, st, true);
    }
    if (g.M <= 16) return gemm8_skinny_launch<1, MODE, OT, false>(g, st, 1);
    if (g.M <= 32 && !(big && small_m_uses_tile(g.M, g.N, g.K))) return gemm8_skinny_launch<2, MODE, OT, false>(g, st, 1);
    if (g.M <= 64 && !(big && small_m_uses_tile(g.M, g.N, g.K))) return gemm8_skinny_launch<4, MODE, OT, false>(g, st, 1);
  }
  {
    if (big) {
      const BigConfig cfg = gemm8_big_config(g.M, g.N, g.K, tiles_256);
      const int bm = cfg.bm;
      int slices = cfg.slices;
      while (slices > 1 && (int64_t)slices * g.M * g.N * 4 > workspace_bytes) slices--;
      if (!workspace || ((uintptr_t)workspace & 15)) slices = 1;
      RAN(bm == 64 ? SGLAMD_KERNEL_TILE64 : bm == 128 ? SGLAMD_KERNEL_TILE128 : bm == 192 ? SGLAMD_KERNEL_TILE192 : SGLAMD_KERNEL_TILE256);
      if (bm == 64) return gemm8_big_launch<MODE, OT, 4, 1>(g, st, slices, workspace);
      if (bm == 128) return gemm8_big_launch<MODE, OT, 4, 2>(g, st, slices, workspace);
      if (bm == 192) return gemm8_big_launch<MODE, OT, 4, 3>(g, st, slices, workspace);
      if (big_wgn() == 2) return gemm8_big_launch<MODE, OT, 2, 4>(g, st, slices, workspace);
      if constexpr (gemm_is_block(MODE)) {
        const bool bias_ok = !out_biased<OT> || (g.N >= 32 && ((uintptr_t)g.bias & 3) == 0);
        if (slices == 1 && wgs > 0 && (wgs & 7) == 0 && bias_ok && gemm8_big_persist_ok(g, wgs)) {
          if constexpr (MODE == GEMM_BLOCK_FP8) {
            if (g.scales_pow2) {
              RAN(SGLAMD_KERNEL_PERSISTENT256_POW2);
              return gemm8_big_persist_launch<MODE, OT, true>(g, st, wgs);
            }
          }
          RAN(SGLAMD_KERNEL_PERSISTENT256);
          return gemm8_big_persist_launch<MODE, OT>(g, st, wgs);
        }
      }
      return gemm8_big_launch<MODE, OT, 4, 4>(g, st, slices, workspace);
    }
  }
  RAN(SGLAMD_KERNEL_GENERIC);
  return gemm8_launch<128, 128, 2, 2, MODE, OT, false>(g, st);
}

// An FP8 linear layer of a few rows in one launch (gemm8_skinny_quantising).
template <int MODE, bool BIASED>
int dispatch_quantising(const GemmArgs& g, int out_dtype, hipStream_t st, bool launch) {
  if (launch) {
    RAN(SGLAMD_KERNEL_STREAMING);
    strip_last_shape = 0;
  }
  if constexpr (BIASED)
    return out_dtype == SGLAMD_BF16 ? gemm8_skinny_quantising<MODE, Biased<BF16>>(g, st, launch)
                                    : gemm8_skinny_quantising<MODE, Biased<F16>>(g, st, launch);
  return out_dtype == SGLAMD_BF16 ? gemm8_skinny_quantising<MODE, BF16>(g, st, launch) : gemm8_skinny_quantising<MODE, F16>(g, st, launch);
}

template <int MODE>
int dispatch_out(const GemmArgs& g, int out_dtype, hipStream_t st, void* ws, int64_t ws_bytes) {
  if (out_dtype == SGLAMD_BF16) return dispatch_dense<MODE, BF16>(g, st, ws, ws_bytes);
  if (out_dtype == SGLAMD_F16) return dispatch_dense<MODE, F16>(g, st, ws, ws_bytes);
  return fail(SGLAMD_EINVAL, "out_dtype must be Half or BFloat16");
}

// The same with a bias: block-scaled modes only (gemm_mode_block_fp8_bias.hip).
template <int MODE>
int dispatch_out_biased(const GemmArgs& g, int out_dtype, hipStream_t st, void* ws, int64_t ws_bytes) {
  if (out_dtype == SGLAMD_BF16) return dispatch_dense<MODE, Biased<BF16>>(g, st, ws, ws_bytes);
  if (out_dtype == SGLAMD_F16) return dispatch_dense<MODE, Biased<F16>>(g, st, ws, ws_bytes);
  return fail(SGLAMD_EINVAL, "out_dtype must be Half or BFloat16");
}

}  // namespace sglamd
