// Fused-MoE tile GEMM for gfx950 where an expert's weights, streamed once from HBM, are the time: a few to about a hundred
// rows per expert.  One workgroup per CU walks the (sorted block, column tile) pairs; its eight waves lie side by side in
// N, each with 32 weight rows of its own and all rows of the block.
//
// Bound by the weight stream, so everything serves it:
//   * a wave's weight rows are read by no other wave: they go to a ring of D stages in LDS that this wave fills and
//     empties at its own pace, and since a block's fragments are taken into registers at its start, its stage is free
//     for block kb + D at once.  The rows of the block, which all waves read, have D + 1 stages, so that one barrier a
//     K block certifies both what has landed and what may be overwritten (gemm8_big_kernel has one per row tile);
//   * the request stream does not stop at a tile's end: it moves on to the next tile D blocks before the products do,
//     the next tile's slot ids, tables, routing weights and scales arriving by direct-to-LDS loads like everything else;
//   * the 32-row tiles behind the last real row are not multiplied;
//   * the weights of an expert with a single block are read once by one workgroup, so they are loaded with the streaming
//     hint and leave the caches to the rows: 512 tokens of the DeepSeek-V3 layer, GEMM 1225 -> 1096 and 683 -> 637 us, with
//     the same 7.5 and 3.8 GB fetched.  An expert's several
//     blocks meet in L2, and with the hint they would not (8 experts, 4096 tokens, persistent walk 1615 -> 1882).
//   * activation scales come in aligned groups of four K blocks (see gemm8_moe_persist_kernel).
// A wave multiplies every row tile with one column tile, so LDS is read for one MFMA pair where gemm8_big_kernel's waves
// read it for two: once the weights are no longer the time, that kernel and its persistent walk win (moe_height_by_rounds).
// Whole layers, us, before -> this kernel: 256 experts of 7168 x 2048, top-8, 128 / 256 / 512 / 1024 / 1536 tokens 1807 ->
// 1644, 2018 -> 1702, 1980 -> 1758, 2160 -> 1849, 2270 -> 1994 (512 tokens by trace: 6.9 and 5.9 TB/s of weights in the two
// GEMMs, matrix pipe 9 and 8 % busy); 64 INT8 experts of 4096 x 1536,
// row scales, top-6, 100 / 250 / 500 / 1000 tokens 249 -> 218, 266 -> 232, 295 -> 251, 334 -> 288.
#pragma once
#include "gemm_big.h"
#include "quant_core.h"

namespace sglamd {

constexpr int GEMM8_MOE_STREAM_MAX_KB = 256;  // 2 column blocks x K blocks: 512 table entries, one load per wave
// K blocks requested ahead of the one being multiplied (what LDS holds)
template <int BM>
constexpr int moe_stream_depth() {
  return BM > 64 ? 2 : 3;
}
template <int BM>
constexpr int moe_stream_smem() {
  constexpr int D = moe_stream_depth<BM>();
  // activation stages | weight stages | activation-scale stages of four K blocks | 256 bytes for loads that must land
  // nowhere | two weight-scale tables | three lists of slot ids | two of routing weights | row maxima of eight waves, or
  // two lists of row scales | eight patches of 32 rows x 64 bytes
  return (D + 1) * BM * 128 + D * 32768 + (D + 1) * BM * 16 + 256 + 2 * 2048 + 3 * BM * 4 + 2 * BM * 4 + 8 * BM * 4 + 8 * 2048;
}

// ACTQ as in gemm8_moe_persist_kernel (g.C the e4m3 rows, g.A16 / g.lda16 their group scales); here a wave's 32 weight rows
// are 16 gate rows and the 16 up rows of the same columns, so that both halves of an output sit in one lane.
template <int MODE, typename OT, int BM, bool ACTQ = false>
__global__ __launch_bounds__(512) void gemm8_moe_stream_kernel(GemmArgs g) {
#if defined(__HIP_DEVICE_COMPILE__)
  static_assert(!ACTQ || MODE == GEMM_BLOCK_FP8, "the fused activation writes e4m3");
  static_assert(BM == 64 || BM == 128, "two or four row tiles");
  constexpr bool BLK = gemm_is_block(MODE);
  constexpr int RT = BM / 32, AL = BM / 64, D = moe_stream_depth<BM>(), BN = 256;
  constexpr int A_STAGE = BM * 128, B_STAGE = BN * 128, S_STAGE = BM * 16;
  constexpr int B_BASE = (D + 1) * A_STAGE, S_BASE = B_BASE + D * B_STAGE, NOWHERE = S_BASE + (D + 1) * S_STAGE;
  constexpr int TBL_BASE = NOWHERE + 256, TBL_BYTES = 2048, IDS_BASE = TBL_BASE + 2 * TBL_BYTES;
  constexpr int WGT_BASE = IDS_BASE + 3 * BM * 4, MAX_BASE = WGT_BASE + 2 * BM * 4, PATCH_BASE = MAX_BASE + 8 * BM * 4;
  constexpr int SAR_BASE = MAX_BASE;  // row modes: two lists of row scales where ACTQ keeps its maxima
  // loads per wave and K block; the scale load of every fourth block comes on top, which makes the waits stricter by one
  constexpr int LPB = AL + 4;
  typedef typename std::conditional<MODE == GEMM_ROW_INT8, v16i, v16f>::type acc16_t;
  typedef typename std::conditional<gemm_is_int8(MODE), v16i, v16f>::type prod16_t;
  static_assert(sizeof(typename OT::storage) == 2, "2-byte outputs");

  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int frow = lane & 31, fk = lane >> 5;

  // tiles of a round and their workgroups: gemm8_moe_persist_kernel's mapping
  const int tiles_n = (g.N + BN - 1) / BN;
  const int nblk = min(g.max_blocks_m, (*g.num_post_pad + BM - 1) / BM);
  const int total = nblk * tiles_n;
  const int nkb = g.K >> 7;
  const int G = (int)gridDim.x;
  const unsigned wpos = (unsigned)xcd_remap((int)blockIdx.x, G);
  auto tile_of_round = [&](int r) -> int { return r * G + (int)((wpos + (unsigned)(r * tiles_n)) % (unsigned)G); };
  int pid = tile_of_round(0);
  if (pid >= total) return;

  const int64_t a_rows = g.num_valid / g.top_k;
  const int half_n = g.N >> 1;

  const uint32_t smem_base = (uint32_t)(uintptr_t)(lds_ptr_t)smem;
  auto descriptor = [](const void* base, int64_t bytes) -> v4i {
    const uint64_t b = (uint64_t)(uintptr_t)base;
    return v4i{(int)(uint32_t)b, (int)((b >> 32) & 0xffff), (int)(bytes < 0x7ffffff0ll ? bytes : 0x7ffffff0ll), 0x00020000};
  };
  // (assembly and five wait states: see gemm8_skinny_kernel)
  auto dma16 = [&](const v4i& rs, uint32_t voff, int soff, uint32_t lds_off, bool nt) {
    if (nt)
      asm volatile("s_nop 4\n\tbuffer_load_dwordx4 %0, %1, %2 offen nt lds" : : "v"(voff), "s"(rs), "s"(soff), "{m0}"(smem_base + lds_off) : "memory");
    else
      asm volatile("s_nop 4\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" : : "v"(voff), "s"(rs), "s"(soff), "{m0}"(smem_base + lds_off) : "memory");
  };
  auto dma4 = [&](const v4i& rs, uint32_t voff, int soff, uint32_t lds_off) {
    asm volatile("s_nop 4\n\tbuffer_load_dword %0, %1, %2 offen lds" : : "v"(voff), "s"(rs), "s"(soff), "{m0}"(smem_base + lds_off) : "memory");
  };
  constexpr uint32_t OUTSIDE = 0x7ffffff0u;

  // ---- the request stream: D blocks ahead of the products, across tiles -----------------------------------------
  uint32_t a_voff[AL], b_voff[2], s_voff = 0;
  v4i a_rs = descriptor(g.A, a_rows * g.lda), b_rs;
  v4i s_rs = descriptor(g.sa, BLK ? ((a_rows - 1) * g.sa_sm + ((nkb + 3) & ~3)) * 4 : 0);
  const int a_len = a_rs[2], s_len = s_rs[2];
  const int w_jump = (ACTQ ? half_n : 16) * (int)g.ldb;  // bytes from a wave's first 16 weight rows to its other 16
  int rot = 0, rk = 0, solo = 0;
  int a_req = 0, w_req = 0, s_req = 0;  // stages of the next request
  const bool rows_mine = wave < BM / 64;  // the waves that fetch one word per slot
  // Tile p, whose slot ids lie in list `ids`, becomes the request stream's tile; its scale tables and the routing weights
  // of its rows are requested into half `b`.
  auto enter = [&](int p, int ids, int b) {
    const bool has = p < total;
    const int pm = has ? p / tiles_n : 0, pn = has ? p - pm * tiles_n : 0;
    const int n0 = pn * (ACTQ ? BN / 2 : BN);
    const int e0 = has ? g.expert_ids[pm] : 0;
    const int ex = __builtin_amdgcn_readfirstlane(max(e0, 0));
    solo = __builtin_amdgcn_readfirstlane((pm == 0 || g.expert_ids[pm - 1] != e0) && (pm + 1 >= nblk || g.expert_ids[pm + 1] != e0) ? 1 : 0);
    a_rs[2] = has ? a_len : 0;
    s_rs[2] = has ? s_len : 0;
    b_rs = descriptor(g.B + (int64_t)ex * g.b_expert_stride, has ? (int64_t)g.N * g.ldb : 0);
    rot = moe_k_rotation(g.ldb, ex, nkb);
    const int* rows = (const int*)(smem + IDS_BASE) + ids * BM;
    auto token = [&](int slot) -> int {  // -1: a padding slot
      const int id = rows[slot];
      return id < g.num_valid ? id / g.top_k : -1;
    };
#pragma unroll
    for (int u = 0; u < AL; u++) {
      const int row = u * 64 + wave * 8 + (lane >> 3);
      const int chunk = (lane & 7) ^ ((row >> 1) & 7);
      const int tok = token(row);
      a_voff[u] = tok >= 0 ? (uint32_t)(tok * (int)g.lda + chunk * 16) : OUTSIDE;
    }
#pragma unroll
    for (int l = 0; l < 2; l++) {
      const int row = (ACTQ ? wave * 16 : wave * 32) + l * 8 + (lane >> 3);
      const int chunk = (lane & 7) ^ ((l * 4 + (lane >> 4)) & 7);
      b_voff[l] = (uint32_t)((n0 + row) * (int)g.ldb + chunk * 16);
    }
    const int slot = min(wave * 64 + lane, BM - 1);
    const int tok = rows_mine ? token(slot) : -1;
    s_voff = tok >= 0 ? (uint32_t)(tok * (int)g.sa_sm) << 2 : OUTSIDE;
    const int e = wave * 64 + lane;
    uint32_t tv;
    int64_t t_bytes;
    if constexpr (BLK) {
      // entry cb * nkb + kb: the scales of column block cb (ACTQ: gate, up) in the order of the walk
      const int cb = e / nkb, kbl = e - cb * nkb + rot, kbb = kbl >= nkb ? kbl - nkb : kbl;
      const int sbrow = ACTQ ? (cb * half_n + n0) >> 7 : min(n0 + cb * 128, g.N - 1) >> 7;
      tv = cb < BN / 128 ? (uint32_t)(sbrow * (int)g.sb_sn + kbb * (int)g.sb_sk) << 2 : OUTSIDE;
      t_bytes = ((int64_t)((g.N - 1) >> 7) * g.sb_sn + (int64_t)(nkb - 1) * g.sb_sk + 1) * 4;
    } else {
      tv = e < BN && n0 + e < g.N ? (uint32_t)((n0 + e) * (int)g.sb_sn) << 2 : OUTSIDE;
      t_bytes = ((int64_t)(g.N - 1) * g.sb_sn + 1) * 4;
    }
    dma4(descriptor(g.sb + (int64_t)ex * g.sb_se, has ? t_bytes : 0), tv, 0, TBL_BASE + b * TBL_BYTES + wave * 256);
    if (g.mul_weight) {
      const int id = rows[slot];
      const uint32_t vo = rows_mine && id < g.num_valid ? (uint32_t)id << 2 : OUTSIDE;
      dma4(descriptor(g.topk_w, (int64_t)g.num_valid * 4), vo, 0, rows_mine ? WGT_BASE + b * BM * 4 + wave * 256 : NOWHERE);
    }
    if constexpr (!BLK) {
      dma4(descriptor(g.sa, ((a_rows - 1) * g.sa_sm + 1) * 4), s_voff, 0,
           rows_mine ? SAR_BASE + b * BM * 4 + wave * 256 : NOWHERE);
    }
    rk = 0;
  };
  // slot ids of tile p's sorted block into list `ids`
  auto request_ids = [&](int p, int ids) {
    dma4(descriptor(g.sorted_ids + (int64_t)(p / tiles_n) * BM, rows_mine ? BM * 4 : 0), (uint32_t)tid << 2, 0,
         rows_mine ? IDS_BASE + ids * BM * 4 + wave * 256 : NOWHERE);
  };
  // where block kb of a walk that starts at block r lies
  auto block_at = [&](int kb, int r) -> int {
    const int k = kb + r - nkb;
    return k + (nkb & (k >> 31));
  };
  // Loads first .. last - 1 of the LPB that make up the next block of the request stream, always issued in this order: the
  // weights, the rows, and with a new group of four blocks its activation scales.
  int kq = 0, nt = 0;
  auto request = [&](int first, int last) {
#pragma unroll
    for (int l = 0; l < LPB; l++) {
      if (l < first || l >= last) continue;
      if (l == 0) {
        kq = block_at(rk, rot);
        nt = solo;
        asm volatile("" : "+s"(nt));  // (see the block loop)
      }
      if (l < 4) {
        const uint32_t vo = b_voff[l & 1] + (uint32_t)(l >> 1) * (uint32_t)w_jump;
        const uint32_t at = B_BASE + w_req * B_STAGE + wave * 4096 + l * 1024;
        if (nt) dma16(b_rs, vo, kq << 7, at, true);
        else dma16(b_rs, vo, kq << 7, at, false);
      } else {
        dma16(a_rs, a_voff[l - 4], kq << 7, a_req * A_STAGE + ((l - 4) * 64 + wave * 8) * 128, false);
      }
      if (l == LPB - 1) {
        if constexpr (BLK) {
          if (rk == 0 || (kq & 3) == 0) {
            if (rows_mine) dma16(s_rs, s_voff, (kq >> 2) << 4, S_BASE + s_req * S_STAGE + wave * 1024, false);
            s_req = s_req == D ? 0 : s_req + 1;
          }
        }
        rk++;
        a_req = a_req == D ? 0 : a_req + 1;
        w_req = w_req == D - 1 ? 0 : w_req + 1;
      }
    }
  };
#define SGLAMD_WAIT_VM(n) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(n) : "memory")

  // ---- fragments -------------------------------------------------------------------------------------------------
  const int fsw = (frow >> 1) & 7;
  int xo[2][2];  // byte offset of chunk c of K half h of row frow
#pragma unroll
  for (int h = 0; h < 2; h++)
#pragma unroll
    for (int c = 0; c < 2; c++) xo[h][c] = (((h * 4 + fk * 2 + c) ^ fsw) << 4) + frow * 128;
  auto frag = [&](const uint8_t* base, int h) -> v8i {
    const v4i lo = *(const v4i*)(base + xo[h][0]);
    const v4i hi = *(const v4i*)(base + xo[h][1]);
    return v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  };
  auto mm_half = [&](const v8i& w, const v8i& x, prod16_t c) -> prod16_t {
    if constexpr (gemm_is_int8(MODE)) {
      const v4i wl = {w[0], w[1], w[2], w[3]}, wh = {w[4], w[5], w[6], w[7]};
      const v4i xl = {x[0], x[1], x[2], x[3]}, xh = {x[4], x[5], x[6], x[7]};
      c = __builtin_amdgcn_mfma_i32_32x32x32_i8(wl, xl, c, 0, 0, 0);
      return __builtin_amdgcn_mfma_i32_32x32x32_i8(wh, xh, c, 0, 0, 0);
    } else {
      return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(w, x, c, 0, 0, 0, 0x7f7f7f7f, 0, 0x7f7f7f7f);
    }
  };

  acc16_t acc[RT];
  prod16_t q[2], zero16;
#pragma unroll
  for (int i = 0; i < RT; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) acc[i][r] = 0;
#pragma unroll
  for (int r = 0; r < 16; r++) q[0][r] = 0, q[1][r] = 0, zero16[r] = 0;
  constexpr int MPH = gemm_is_int8(MODE) ? 2 : 1, FOLDN = gemm_is_int8(MODE) ? 32 : 16;  // instructions of mm_half, fold
  float sc = 0.f, sc1 = 0.f;  // scales of the product that waits to be folded (ACTQ: of its gate and its up half)
  auto fold = [&](acc16_t& dst, const prod16_t& p) {
    if constexpr (BLK) {
#pragma unroll
      for (int r = 0; r < 16; r++) dst[r] = fmaf((float)p[r], ACTQ && r >= 8 ? sc1 : sc, dst[r]);
    }
  };

  // ---- the first tile ----------------------------------------------------------------------------------------------
  {
    const int pm = pid / tiles_n;
    if (tid < BM) ((int*)(smem + IDS_BASE))[tid] = g.sorted_ids[(int64_t)pm * BM + tid];
    __syncthreads();
    enter(pid, 0, 0);
#pragma unroll
    for (int d = 0; d < D; d++) request(0, LPB);
    SGLAMD_WAIT_VM((D - 1) * LPB);
    __syncthreads();
  }
  int round = 0, list = 0, buf = 0, rot_now = rot;
  int a_cur = 0, w_cur = 0, s_cur = 0;
  // 32-row tiles up to the last one that holds a real row of the sorted block in list `l`: the sort puts them first, a caller's
  // own lists need not
  auto live_tiles = [&](int l) -> int {
    const int* rows = (const int*)(smem + IDS_BASE) + l * BM;
    int live = 1;
#pragma unroll
    for (int u = 0; u < BM / 64; u++) {
      const uint64_t real = __ballot(rows[u * 64 + lane] < g.num_valid);
      if (real) live = u * 2 + (real >> 32 ? 2 : 1);
    }
    return __builtin_amdgcn_readfirstlane(live);
  };
  int live_now = live_tiles(0);
  // What a block needs first is fetched under the last products of the block before: its weights, the fragments and scales
  // of its last two live row tiles (by the parity of the tile) and its weight scales.
  v8i wf0, wf1, x[2][2];
  float sa[2] = {1.f, 1.f}, sbv = 1.f, sbv1 = 1.f;
  auto scale_at = [&](int stage, int k, int t) -> float {
    return ((const float*)(smem + S_BASE + stage * S_STAGE))[(t * 32 + frow) * 4 + (k & 3)];
  };
  auto fetch_x = [&](int p, int h, int stage, int s_stage, int k, int tiles) {
    const int t = p == 0 ? (tiles - 1) & ~1 : max(1, (tiles & ~1) - 1);
    x[p][h] = frag(smem + stage * A_STAGE + t * 4096, h);
    if (BLK && h == 1) sa[p] = scale_at(s_stage, k, t);
  };
  auto fetch_w = [&](int stage, int h) { (h ? wf1 : wf0) = frag(smem + B_BASE + stage * B_STAGE + wave * 4096, h); };
  const int my_scale = ACTQ ? 0 : (wave >> 2) * nkb;
  auto fetch_scale = [&](int b, int kb, float& s0, float& s1) {
    if constexpr (BLK) {
      const float* tbl = (const float*)(smem + TBL_BASE + b * TBL_BYTES);
      s0 = tbl[my_scale + kb];
      if constexpr (ACTQ) s1 = tbl[nkb + kb];
    }
  };
  fetch_w(0, 0);
  fetch_w(0, 1);
#pragma unroll
  for (int p = 0; p < 2; p++) {
    fetch_x(p, 0, 0, 0, rot_now, live_now);
    fetch_x(p, 1, 0, 0, rot_now, live_now);
  }
  fetch_scale(0, 0, sbv, sbv1);

  for (;;) {
    const int next = tile_of_round(round + 1);
    const bool has_next = next < total;
    const int pm = pid / tiles_n, n0 = (pid - pm * tiles_n) * (ACTQ ? BN / 2 : BN);
    const int expert = __builtin_amdgcn_readfirstlane(g.expert_ids[pm]);
    const int* rows = (const int*)(smem + IDS_BASE) + list * BM;
    const int list_next = list == 2 ? 0 : list + 1;
    int live_next = 1;
    if (has_next) request_ids(next, list_next);

    for (int kb = 0; kb < nkb; kb++) {
      const uint8_t* xs = smem + a_cur * A_STAGE;
      const int k_now = block_at(kb, rot_now);
      // (invariants of the loop, or functions of its counter, to the compiler, which would clone the loop for their values)
      int live = __builtin_amdgcn_readfirstlane(live_now), left = __builtin_amdgcn_readfirstlane(nkb - kb);
      int tile_then = __builtin_amdgcn_readfirstlane(next);
      asm volatile("" : "+s"(live), "+s"(left), "+s"(tile_then));
      // this block's weights are in registers (the statement waits for them): their stage takes block kb + D
      asm volatile("" : "+v"(wf0), "+v"(wf1) : : "memory");
      if (left == D) {
        enter(tile_then, list_next, buf ^ 1);
        live_next = tile_then < total ? live_tiles(list_next) : 1;
      }
      // Eight waves that issue a block's loads at once park the CU's vector memory pipe (16 cycles a load) with idle matrix
      // pipes, so the steps carry some each; those of the steps that are not run go out here.
      if constexpr (RT > 2) {
        if (live <= 3) request(0, 2);
        if (live <= 2) request(2, 4);
      } else {
        request(0, 2);
      }
      fold(acc[0], q[0]);
      sc = sc1 = 0.f;
      int live_then = live;  // live tiles, scale stage and place of the block behind this one
      int s_then = s_cur, k_then = 0;
      // row tiles from the last live one down to the first, each folded under the products of the next
      auto step = [&](auto tile_c) {
        constexpr int i = decltype(tile_c)::value, p = i & 1;
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (BLK) q[p] = mm_half(wf0, x[p][0], zero16);
        else acc[i] = mm_half(wf0, x[p][0], acc[i]);
        __builtin_amdgcn_sched_group_barrier(0x8, MPH, 0);
        if constexpr (i > 1) {
          x[p][0] = frag(xs + (i - 2) * 4096, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        } else {
          if constexpr (i == 0) fetch_w(w_cur, 0);
          fetch_x(p, 0, a_cur, s_then, k_then, live_then);
          __builtin_amdgcn_sched_group_barrier(0x100, i == 0 ? 4 : 2, 0);
        }
        if constexpr (BLK && i + 1 < RT) {
          fold(acc[i + 1], q[p ^ 1]);
          __builtin_amdgcn_sched_group_barrier(0x2, FOLDN, 0);
        }
        if constexpr (BLK) q[p] = mm_half(wf1, x[p][1], q[p]);
        else acc[i] = mm_half(wf1, x[p][1], acc[i]);
        __builtin_amdgcn_sched_group_barrier(0x8, MPH, 0);
        if constexpr (BLK) {
          sc = sa[p] * sbv;
          if constexpr (ACTQ) sc1 = sa[p] * sbv1;
        }
        if constexpr (i > 1) {
          x[p][1] = frag(xs + (i - 2) * 4096, 1);
          if constexpr (BLK) sa[p] = scale_at(s_cur, k_now, i - 2);
        } else {
          if constexpr (i == 0) fetch_w(w_cur, 1);
          fetch_x(p, 1, a_cur, s_then, k_then, live_then);
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (i == 3) request(0, 2);
        if constexpr (i == 2) request(2, 4);
      };
      if constexpr (RT > 3) if (live > 3) step(std::integral_constant<int, 3>{});
      if constexpr (RT > 2) if (live > 2) step(std::integral_constant<int, 2>{});
      // Block kb + 1 has landed here (requested D - 1 blocks ago) and, behind the barrier, everywhere.  The fragments of the
      // two tiles that are left are in registers, so every wave is past its reads of this block's activation stage: the
      // next block's request takes it.  Loads issued since block kb + 1's: those of D - 2 whole blocks and what this block
      // has requested so far.
      SGLAMD_WAIT_VM((D - 2) * LPB + (RT > 2 ? 4 : 2));
      __builtin_amdgcn_s_barrier();
      asm volatile("" : : : "memory");
      request(RT > 2 ? 4 : 2, LPB);
      a_cur = a_cur == D ? 0 : a_cur + 1;
      w_cur = w_cur == D - 1 ? 0 : w_cur + 1;
      const bool last = left == 1;
      live_then = last ? live_next : live;
      k_then = last ? rot : block_at(nkb - left + 1, rot_now);
      if (last || (k_then & 3) == 0) s_then = s_cur == D ? 0 : s_cur + 1;
      float sbv_n, sbv1_n;
      fetch_scale(last ? buf ^ 1 : buf, last ? 0 : nkb - left + 1, sbv_n, sbv1_n);
      if (live > 1) {
        step(std::integral_constant<int, 1>{});
      } else if (live_then > 1) {
        fetch_x(1, 0, a_cur, s_then, k_then, live_then);
        fetch_x(1, 1, a_cur, s_then, k_then, live_then);
      }
      step(std::integral_constant<int, 0>{});
      sbv = sbv_n;
      sbv1 = sbv1_n;
      s_cur = s_then;
    }
    fold(acc[0], q[0]);
    sc = sc1 = 0.f;

    // ---- the finished tile leaves; the next one's first D blocks are on their way ---------------------------------
    const float* wgts = (const float*)(smem + WGT_BASE) + buf * BM;
    const v4i c_rs = descriptor(g.C, (int64_t)g.num_valid * g.ldc * (ACTQ ? 1 : 2));
    if constexpr (ACTQ) {
      // the roundings and the quantisation of gemm8_moe_persist_kernel
      float* s_max = (float*)(smem + MAX_BASE);
      const float wgt = expert < 0 ? 0.f : 1.f;
#pragma unroll
      for (int i = 0; i < RT; i++) {
        if (i >= live_now) break;
        float m = 0.f;
#pragma unroll
        for (int r = 0; r < 8; r++) {
          const float gv = OT::to_f32(OT::from_f32(acc[i][r] * wgt));
          const float uv = OT::to_f32(OT::from_f32(acc[i][r + 8] * wgt));
          const float sv = silu_rounded<OT>(gv);
          const float y = OT::to_f32(OT::from_f32(sv * uv));
          acc[i][r] = y;
          m = fmaxf(m, fabsf(y));
        }
        m = fmaxf(m, __shfl_xor(m, 32, 64));
        if (fk == 0) s_max[wave * BM + i * 32 + frow] = m;
      }
      asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" : : : "memory");
      uint8_t* out = smem + PATCH_BASE;  // [BM] rows of 128 bytes, 16-byte pieces swizzled with the row
#pragma unroll
      for (int i = 0; i < RT; i++) {
        if (i >= live_now) break;
        const int trow = i * 32 + frow;
        float amax = 1e-10f;
#pragma unroll
        for (int w = 0; w < 8; w++) amax = fmaxf(amax, s_max[w * BM + trow]);
        const float mul = 448.f / amax;
#pragma unroll
        for (int rq = 0; rq < 2; rq++) {
          const uint32_t w = pack4_e4m3(clampf(acc[i][rq * 4] * mul, -448.f, 448.f), clampf(acc[i][rq * 4 + 1] * mul, -448.f, 448.f),
                                        clampf(acc[i][rq * 4 + 2] * mul, -448.f, 448.f), clampf(acc[i][rq * 4 + 3] * mul, -448.f, 448.f));
          *(uint32_t*)(out + trow * 128 + ((wave ^ (trow & 7)) << 4) + rq * 8 + fk * 4) = w;
        }
        const int mine = rows[trow];
        if (wave == 0 && fk == 0 && mine < g.num_valid)
          ((float*)g.A16)[(int64_t)mine * g.lda16 + (n0 >> 7)] = amax * (1.0f / 448.f);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" : : : "memory");
#pragma unroll
      for (int u = 0; u < AL; u++) {
        const int row = (wave * AL + u) * 8 + (lane >> 3), piece = lane & 7;
        const v4i v = *(const v4i*)(out + row * 128 + ((piece ^ (row & 7)) << 4));
        const int m = rows[row];
        const uint32_t vo = m < g.num_valid ? (uint32_t)(m * (int)g.ldc + n0 + piece * 16) : 0xfffffff0u;
        // (s_nop 4 and s_nop 1: see gemm8_moe_persist_kernel)
        asm volatile("s_nop 4\n\tbuffer_store_dwordx4 %0, %1, %2, 0 offen\n\ts_nop 1" : : "v"(v), "v"(vo), "s"(c_rs) : "memory");
      }
    } else {
      uint8_t* stg = smem + PATCH_BASE + wave * 2048;  // 32 rows of 64 bytes, 16-byte pieces swizzled with the row
      float sbn[16];
      if constexpr (!BLK) {
#pragma unroll
        for (int rq = 0; rq < 4; rq++) {
          const v4f s4 = *(const v4f*)((const float*)(smem + TBL_BASE + buf * TBL_BYTES) + wave * 32 + 8 * rq + 4 * fk);
#pragma unroll
          for (int r = 0; r < 4; r++) sbn[rq * 4 + r] = s4[r];
        }
      }
#pragma unroll
      for (int i = 0; i < RT; i++) {
        if (i >= live_now) break;
        const float wgt = expert < 0 ? 0.f : g.mul_weight ? wgts[i * 32 + frow] : 1.f;
        float sam = 1.f;
        if constexpr (!BLK) sam = ((const float*)(smem + SAR_BASE))[buf * BM + i * 32 + frow];
        float v[16];
#pragma unroll
        for (int r = 0; r < 16; r++) {
          if constexpr (BLK) v[r] = acc[i][r] * wgt;
          else if constexpr (MODE == GEMM_ROW_FP8) v[r] = acc[i][r] * sbn[r] * sam * wgt;
          else v[r] = (float)acc[i][r] * (sbn[r] * sam) * wgt;
        }
#pragma unroll
        for (int rq = 0; rq < 4; rq++) {
          const v2i w = {(int)OT::pack2(v[rq * 4], v[rq * 4 + 1]), (int)OT::pack2(v[rq * 4 + 2], v[rq * 4 + 3])};
          *(v2i*)(stg + frow * 64 + ((rq ^ ((frow >> 2) & 3)) << 4) + fk * 8) = w;
        }
#pragma unroll
        for (int half = 0; half < 2; half++) {
          const int row = (lane >> 2) + 16 * half, piece = lane & 3;
          const v4i o = *(const v4i*)(stg + row * 64 + ((piece ^ ((row >> 2) & 3)) << 4));
          const int m = rows[i * 32 + row];
          const int n = n0 + wave * 32 + piece * 8;
          const uint32_t vo = m < g.num_valid && n < g.N ? (uint32_t)((m * (int)g.ldc + n) * 2) : 0xfffffff0u;
          asm volatile("s_nop 4\n\tbuffer_store_dwordx4 %0, %1, %2, 0 offen\n\ts_nop 1" : : "v"(o), "v"(vo), "s"(c_rs) : "memory");
        }
      }
    }
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][r] = 0;
#pragma unroll
    for (int r = 0; r < 16; r++) q[0][r] = 0;
    if (!has_next) break;
    pid = next;
    round++;
    live_now = live_next;
    list = list_next;
    buf ^= 1;
    rot_now = rot;
  }
  // the trailing empty-range loads still write LDS: none may be in flight when the workgroup ends
  __builtin_amdgcn_s_waitcnt(0x0070);
#undef SGLAMD_WAIT_VM
#endif
}

// Shapes the kernel takes: whole K blocks, enough of them that a tile's ids and tables land under the tile in front of it,
// 32-bit buffer offsets, whole aligned 16-byte output pieces, no bias, block modes with scales in whole groups.
template <int BM>
static inline bool gemm8_moe_stream_ok(const GemmArgs& g, bool block) {
  const int nkb = g.K >> 7;
  return (g.K % 128) == 0 && nkb >= 2 * moe_stream_depth<BM>() && nkb <= GEMM8_MOE_STREAM_MAX_KB && (g.N & 7) == 0 &&
         (g.ldc & 7) == 0 && (((uintptr_t)g.C) & 15) == 0 && !g.bias && (int64_t)g.num_valid * g.ldc * 2 < 0x7fffffffll &&
         (int64_t)(g.num_valid / g.top_k) * g.lda < 0x7ffffff0ll && (int64_t)(g.N + 255) * g.ldb < 0x7ffffff0ll &&
         (!block || moe_quad_scales(g));
}

template <int MODE, typename OT, int BM, bool ACTQ = false>
static int gemm8_moe_stream_launch(const GemmArgs& g, hipStream_t st) {
  auto kern = gemm8_moe_stream_kernel<MODE, OT, BM, ACTQ>;
  constexpr int smem = moe_stream_smem<BM>();
  static_assert(smem <= 160 * 1024, "LDS of a CU");
  static SmemAttrOnce attr;
  hipError_t e = raise_dynamic_smem(attr, (const void*)kern, smem);
  if (e != hipSuccess) return fail(SGLAMD_EHIP, "hipFuncSetAttribute: %s", hipGetErrorString(e));
  const int64_t tiles = (int64_t)((g.N + 255) / 256) * g.max_blocks_m;
  if (tiles <= 0) return SGLAMD_OK;
  const int64_t wgs = tiles < device_cus() ? tiles : device_cus();
  hipLaunchKernelGGL(kern, dim3((unsigned)wgs), dim3(512), smem, st, g);
  return check_launch("gemm8_moe_stream");
}

}  // namespace sglamd
