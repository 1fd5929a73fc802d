// Weight-streaming GEMM for 17 to 128 activation rows (up to 32 of them for weights past 100 MB): every workgroup owns all rows and up to 128 or 160 weight rows, and
// walks (K slice, column tile) items one after the other.
//
// What bounds these calls is how many bytes a CU takes in, weights from HBM and activation rows from L2 alike (about 34 KB a
// microsecond with all CUs at it), and how much of a K block's time a wave spends on anything but products.  Hence:
//   * loading and multiplying are different waves.  A wave issues one direct-to-LDS load in 50 cycles at best; with a
//     wave's products behind its own loads, fragment reads and barrier, a K block of 128 x 160 took it 2200 cycles for 512
//     cycles of products.  Eight waves, NS of them with a strip of 32 weight rows each and 8 - NS that only load: the
//     chain of a multiplying wave is 1200 cycles, and the loaders are never behind a product;
//   * the request stream runs on across items (loaders know nothing of outputs), so an item's start costs no ramp;
//   * one barrier a K block: by then every fragment of the block is in registers and the next block has landed;
//   * tiles of any multiple of 16 weight rows, so that the items fill the chip: 36864 weight rows are 256 tiles of 144 where
//     the tile kernel has 144 tiles of 256 for 256 CUs.
// Kernel alone under the tracer, us, tile kernel (64 rows: wide streaming form) -> this, cold weights: 36864 x 7168 at 64 / 96 / 128 rows
// 51 / 66 / 69 -> 46 / 49 / 56 (in a graph, weights in turn: 44 / - / 55 to 59 with the clock; with the quantiser in front 47 / 52 / 57);
// 57344 x 8192 at 128 rows 113 -> 100.  At 128 rows the loaders alone, without a product, need 46: the rest is the clock (1.75 to 1.9 GHz
// under load) and the fragment reads.  Not faster, and not kept: the loads spread over the multiplying waves (61 at 128 rows), two waves
// to a strip with half of the rows each (69), four stages instead of three, a fragment copy per row tile (spills), weight rows at another
// pitch (only multiples of 4096 bytes matter, see `rotate`).
#pragma once
#include "gemm_big.h"

namespace sglamd {

constexpr int STRIP_MAX_ROWS = 128;  // activation rows
// Stages: what LDS holds.  Up to 32 rows, where a block takes the multiplying waves little, the blocks in flight are what keeps HBM
// busy (36864 x 7168 at 32 rows: streaming kernel 51, three stages 48, five 45 us); else three are as good as four.
template <int RT, int NS>
constexpr int strip_stages() {
  return RT > 1 ? 3 : NS == 3 ? 8 : NS == 4 ? 6 : 5;
}
constexpr int STRIP_MAX_KB = 256;  // K blocks of a slice: what a row of the scale table holds

// One K block in LDS: weights, rows, row scales
template <int MODE, int RT, int NS>
constexpr int strip_stage() {
  return NS * 4096 + RT * 4096 + (gemm_is_block(MODE) ? (RT + 1) / 2 * 256 : 0);
}
// the stages, a patch of 32 rows x 64 bytes per multiplying wave, two tables of three rows of weight scales (see strip_tables_hold)
template <int MODE, int RT, int NS>
constexpr int strip_smem() {
  return strip_stages<RT, NS>() * strip_stage<MODE, RT, NS>() + NS * 2048 + (gemm_is_block(MODE) ? 2 * 3 * STRIP_MAX_KB * 4 : 0);
}

// RT row tiles of 32, NS strips of 32 weight rows.  g.rows_per_wg: weight rows of a tile (a multiple of 16); g.max_blocks_m: K slices
// (more than one: g.C is a [slices, M, N] fp32 workspace); g.streams: weights past the caches.
template <int MODE, typename OT, int RT, int NS>
__global__ __launch_bounds__(512) void gemm8_strip_kernel(GemmArgs g) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr bool BLK = gemm_is_block(MODE);
  constexpr int D = strip_stages<RT, NS>(), NL = 8 - NS;
  // wave-wide loads of a K block: groups of eight weight rows, of eight rows, of 64 row scales; loading wave l issues l, l + NL, ...
  constexpr int WG = 4 * NS, AG = 4 * RT, SG = BLK ? (RT + 1) / 2 : 0, UNITS = WG + AG + SG;
  constexpr int LPB = (UNITS + NL - 1) / NL;
  constexpr int STAGE = strip_stage<MODE, RT, NS>(), A_OFF = WG * 1024, S_OFF = A_OFF + AG * 1024;
  constexpr int PATCH_BASE = D * STAGE, TBL_BASE = PATCH_BASE + NS * 2048, TBL_BYTES = 3 * STRIP_MAX_KB * 4;
  static_assert(RT >= 1 && RT <= 4, "fragments of two row tiles, by the parity of the tile");
  static_assert((D - 1) * LPB < 64, "vmcnt field is 6 bits");
  typedef typename std::conditional<MODE == GEMM_ROW_INT8, v16i, v16f>::type acc16_t;
  typedef typename std::conditional<gemm_is_int8(MODE), v16i, v16f>::type prod16_t;
  typedef typename OT::storage OS;
  static_assert(sizeof(OS) == 2, "2-byte outputs");

  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  const int R = g.rows_per_wg, slices = g.max_blocks_m;
  const int tiles_n = (g.N + R - 1) / R, items = tiles_n * slices, G = (int)gridDim.x;
  const int nkb_all = (g.K + 127) >> 7;
  // item: slice by slice, the column tiles of each
  auto k_first = [&](int slice) -> int { return __builtin_amdgcn_readfirstlane(nkb_all * slice / slices); };
  // Column tiles start their walk at different K blocks where the weight rows' pitch would put the same block of all rows on a
  // few memory channels (see moe_k_rotation): 65536 x 4096 at 128 rows 72 -> 56 us, other pitches unchanged.
  const bool rotate = !(g.ldb & 4095);
  const int first = xcd_remap((int)blockIdx.x, G);

  if (wave >= NS) {
    // ---- loading waves ---------------------------------------------------------------------------------------------
    const int loader = wave - NS;
    __builtin_amdgcn_s_setprio(3);
    const uint32_t smem_base = (uint32_t)(uintptr_t)(lds_ptr_t)smem;
    constexpr uint32_t OUTSIDE = 0x7ffffff0u;
    auto descriptor = [](const void* base, int64_t bytes) -> v4i {
      const uint64_t b = (uint64_t)(uintptr_t)base;
      // (a minimum of 64-bit values is computed by the vector unit)
      return v4i{__builtin_amdgcn_readfirstlane((int)(uint32_t)b), __builtin_amdgcn_readfirstlane((int)((b >> 32) & 0xffff)),
                 __builtin_amdgcn_readfirstlane((int)(bytes < 0x7ffffff0ll ? bytes : 0x7ffffff0ll)), 0x00020000};
    };
    auto dma16 = [&](const v4i& rs, uint32_t voff, int soff, uint32_t lds_off) {
      asm volatile("s_nop 4\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" : : "v"(voff), "s"(rs), "s"(soff), "{m0}"(smem_base + lds_off) : "memory");
    };
    auto dma16_nt = [&](const v4i& rs, uint32_t voff, int soff, uint32_t lds_off) {
      asm volatile("s_nop 4\n\tbuffer_load_dwordx4 %0, %1, %2 offen nt lds" : : "v"(voff), "s"(rs), "s"(soff), "{m0}"(smem_base + lds_off) : "memory");
    };
    auto dma4 = [&](const v4i& rs, uint32_t voff, int soff, uint32_t lds_off) {
      asm volatile("s_nop 4\n\tbuffer_load_dword %0, %1, %2 offen lds" : : "v"(voff), "s"(rs), "s"(soff), "{m0}"(smem_base + lds_off) : "memory");
    };
    const v4i a_rs = descriptor(g.A, (int64_t)g.M * g.lda), b_rs = descriptor(g.B, (int64_t)g.N * g.ldb);
    const v4i s_rs = descriptor(g.sa, BLK ? ((int64_t)(g.M - 1) * g.sa_sm + (int64_t)(nkb_all - 1) * g.sa_sk + 1) * 4 : 0);
    const bool nt = g.streams > 0;
    // row modes: K need not fill its last block, whose pieces past the end of a row are requested out of range (zeros; a row's
    // neighbour may hold NaN).  Whether the lane's piece is one of them, by the parity of the group of rows.
    bool dead[2] = {};
    if constexpr (!BLK) {
      if (g.K & 127) {
#pragma unroll
        for (int l = 0; l < 2; l++) dead[l] = ((lane & 7) ^ ((l * 4 + (lane >> 4)) & 7)) >= (g.K & 127) >> 4;
      }
    }

    // the request stream: block `rk` of item `at`
    uint32_t voff[LPB];
    int at = first, rk = 0, r_nkb = 0, r_begin = 0, r_rot = 0, r_stage = 0, r_buf = 0;
    auto enter = [&]() {
      const int slice = __builtin_amdgcn_readfirstlane(at / tiles_n), pn = at - slice * tiles_n;
      const int n0 = pn * R, n_end = min(n0 + R, (int)g.N);
      r_begin = k_first(slice);
      r_nkb = k_first(slice + 1) - r_begin;
      r_rot = rotate ? __builtin_amdgcn_readfirstlane((int)((unsigned)(pn * 5) % (unsigned)r_nkb)) : 0;
      rk = 0;
#pragma unroll
      for (int u = 0; u < LPB; u++) {
        const int e = u * NL + loader;
        const int row = (e < WG ? e : e - WG) * 8 + (lane >> 3), chunk = (lane & 7) ^ ((row >> 1) & 7);
        const int srow = min(max(e - WG - AG, 0) * 64 + lane, (int)g.M - 1);
        if (e < WG) voff[u] = n0 + row < n_end ? (uint32_t)((n0 + row) * (int)g.ldb + chunk * 16) : OUTSIDE;
        else if (e < WG + AG) voff[u] = row < g.M ? (uint32_t)(row * (int)g.lda + chunk * 16) : OUTSIDE;
        else voff[u] = (uint32_t)(srow * (int)g.sa_sm) << 2;
      }
      if constexpr (BLK) {
        // weight scales of the tile's column blocks (at most three), in the order of the walk
        const int nb0 = n0 >> 7, nbs = ((n_end - 1) >> 7) - nb0 + 1, chunks = (r_nkb + 63) >> 6;
        const int64_t span = ((int64_t)(nkb_all - 1) * g.sb_sk + 1) * 4;
        for (int c = loader; c < nbs * chunks; c += NL) {
          const int cb = __builtin_amdgcn_readfirstlane(c / chunks), kb = (c - cb * chunks) * 64 + lane;
          int kbr = kb + r_rot;
          if (kbr >= r_nkb) kbr -= r_nkb;
          dma4(descriptor(g.sb + (int64_t)__builtin_amdgcn_readfirstlane(nb0 + cb) * g.sb_sn, span), kb < r_nkb ? (uint32_t)((r_begin + kbr) * (int)g.sb_sk) << 2 : OUTSIDE, 0,
               __builtin_amdgcn_readfirstlane(TBL_BASE + r_buf * TBL_BYTES + (cb * STRIP_MAX_KB + (c - cb * chunks) * 64) * 4));
        }
        r_buf ^= 1;
      }
    };
    auto request = [&]() {  // the next block of the stream, if there is one
      if (at >= items) return;
      if (rk == r_nkb) {
        at += G;
        if (at >= items) return;
        enter();
      }
      int kq = rk + r_rot;
      if (kq >= r_nkb) kq -= r_nkb;
      kq = __builtin_amdgcn_readfirstlane(kq + r_begin);
      const int stage = __builtin_amdgcn_readfirstlane(r_stage * STAGE);
      const bool tail = !BLK && kq == nkb_all - 1;
#pragma unroll
      for (int u = 0; u < LPB; u++) {
        const int e = u * NL + loader;
        const uint32_t to = (uint32_t)(stage + e * 1024), vo = tail && dead[e & 1] ? OUTSIDE : voff[u];
        if (u * NL + NL <= WG || e < WG) {
          if (nt) dma16_nt(b_rs, vo, kq << 7, to);
          else dma16(b_rs, vo, kq << 7, to);
        } else if (u * NL + NL <= WG + AG || e < WG + AG) {
          dma16(a_rs, vo, kq << 7, to);
        } else if (u * NL + NL <= UNITS || e < UNITS) {
          dma4(s_rs, voff[u], (kq * (int)g.sa_sk) << 2, (uint32_t)(stage + S_OFF + (e - WG - AG) * 256));
        }
      }
      rk++;
      r_stage = r_stage == D - 1 ? 0 : r_stage + 1;
    };
    const bool full = UNITS % NL == 0 || (LPB - 1) * NL + loader < UNITS;  // issues LPB loads a block, not one less
    // all but the last `blocks` blocks requested (at most `most`, a constant) have landed
    auto landed = [&](int blocks, auto most) {
#pragma unroll
      for (int d = decltype(most)::value; d >= 0; d--)
        if (blocks == d) {
          if (full) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(d * LPB) : "memory");
          else asm volatile("s_waitcnt vmcnt(%0)" : : "n"(d * (LPB - 1)) : "memory");
        }
    };
    int left = 0;  // blocks of this workgroup's items
    for (int it = first; it < items; it += G) {
      const int slice = __builtin_amdgcn_readfirstlane(it / tiles_n);
      left += k_first(slice + 1) - k_first(slice);
    }
    enter();
    for (int d = 0; d < D; d++) request();
    left = __builtin_amdgcn_readfirstlane(left);
    landed(min(left, D) - 1, std::integral_constant<int, D - 1>{});
    __builtin_amdgcn_s_barrier();
    for (; left > 0; left--) {
      // the next block has landed; behind the barrier this one is in the multiplying waves' registers, and its stage is free
      landed(max(min(left, D) - 2, 0), std::integral_constant<int, D - 2>{});
      __builtin_amdgcn_s_barrier();
      request();
    }
    return;
  }

  // ---- multiplying waves: one strip of 32 weight rows each ------------------------------------------------------------
  const int frow = lane & 31, fk = lane >> 5;
  const int fsw = (frow >> 1) & 7;
  const uint8_t* fb[2][2];  // chunk c of K half h of row frow
#pragma unroll
  for (int h = 0; h < 2; h++)
#pragma unroll
    for (int c = 0; c < 2; c++) fb[h][c] = smem + ((((h * 4 + fk * 2 + c) ^ fsw) << 4) + frow * 128);
  auto frag = [&](int at, int h) -> v8i {
    const v4i lo = *(const v4i*)(fb[h][0] + at);
    const v4i hi = *(const v4i*)(fb[h][1] + at);
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
  constexpr int NQ = RT == 3 ? 3 : 2;  // products that wait to be folded: a tile's and the one's before, never the same registers
  auto qi = [](int tile) constexpr { return RT == 3 ? tile : tile & 1; };
  acc16_t acc[RT];
  prod16_t q[NQ], zero16;
#pragma unroll
  for (int i = 0; i < RT; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) acc[i][r] = 0;
#pragma unroll
  for (int r = 0; r < 16; r++) q[0][r] = 0, zero16[r] = 0;
  constexpr int MPH = gemm_is_int8(MODE) ? 2 : 1, FOLDN = gemm_is_int8(MODE) ? 32 : 16;
  float sc = 0.f, sc1 = 0.f;
  auto fold = [&](acc16_t& dst, const prod16_t& p) {
    if constexpr (BLK) {
#pragma unroll
      for (int r = 0; r < 16; r++) dst[r] = fmaf((float)p[r], r >= 8 ? sc1 : sc, dst[r]);
    }
  };
  auto row_scale = [&](int stage, int t) -> float { return *(const float*)(smem + stage + S_OFF + (t * 32 + frow) * 4); };
  // weight scales of the strip's two halves of 16 columns, which may lie in two blocks of 128
  const float *sb0 = nullptr, *sb1 = nullptr;
  auto tables = [&](int item, int buf, const float*& t0, const float*& t1) {
    const int pn = item - __builtin_amdgcn_readfirstlane(item / tiles_n) * tiles_n, n0 = pn * R, last = min(n0 + R, (int)g.N) - 1;
    const float* tbl = (const float*)(smem + TBL_BASE + buf * TBL_BYTES);
    t0 = tbl + ((min(n0 + wave * 32, last) >> 7) - (n0 >> 7)) * STRIP_MAX_KB;
    t1 = tbl + ((min(n0 + wave * 32 + 16, last) >> 7) - (n0 >> 7)) * STRIP_MAX_KB;
  };
  tables(first, 0, sb0, sb1);

  __builtin_amdgcn_s_barrier();  // block 0 has landed
  asm volatile("" : : : "memory");
  int st = 0, buf = 0;
  float sbv = 1.f, sbv1 = 1.f;
  if constexpr (BLK) sbv = sb0[0], sbv1 = sb1[0];
  // fragments of two row tiles, by the parity of the tile; tiles go from the last one down
  v8i wf[2], x[2][2];
  float sa[2];
  constexpr int T1 = RT - 1, T2 = RT > 1 ? RT - 2 : 0;
#pragma unroll
  for (int h = 0; h < 2; h++) {
    wf[h] = frag(wave * 4096, h);
    x[T1 & 1][h] = frag(A_OFF + T1 * 4096, h);
    x[T2 & 1][h] = frag(A_OFF + T2 * 4096, h);
  }
  sa[T1 & 1] = BLK ? row_scale(0, T1) : 1.f;
  sa[T2 & 1] = BLK ? row_scale(0, T2) : 1.f;

  for (int item = first; item < items; item += G) {
    const int slice = __builtin_amdgcn_readfirstlane(item / tiles_n), pn = item - slice * tiles_n;
    const int nkb = k_first(slice + 1) - k_first(slice);
    const float *sb0_next = sb0, *sb1_next = sb1;
    if (item + G < items) tables(item + G, buf ^ 1, sb0_next, sb1_next);
    for (int kb = 0; kb < nkb; kb++) {
      const int now = st * STAGE, st_next = st == D - 1 ? 0 : st + 1, then = st_next * STAGE;
      float sbv_n = 1.f, sbv1_n = 1.f;
      if constexpr (RT == 1) {
        // one tile: the next block's fragments are read while the products are on their way, and these are folded behind that
        if constexpr (BLK) q[0] = mm_half(wf[1], x[0][1], mm_half(wf[0], x[0][0], zero16));
        else acc[0] = mm_half(wf[1], x[0][1], mm_half(wf[0], x[0][0], acc[0]));
        sc = sa[0] * sbv;
        sc1 = sa[0] * sbv1;
        __builtin_amdgcn_sched_barrier(0);
        // (as below: the products, which the compiler may put behind the barrier, do not wait for the fragments in front of it)
        asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" : : : "memory");
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int h = 0; h < 2; h++) {
          wf[h] = frag(then + wave * 4096, h);
          x[0][h] = frag(then + A_OFF, h);
        }
        if constexpr (BLK) {
          const bool last = kb + 1 == nkb;
          sa[0] = row_scale(then, 0);
          sbv = *(last ? sb0_next : sb0 + kb + 1);
          sbv1 = *(last ? sb1_next : sb1 + kb + 1);
        }
        __builtin_amdgcn_sched_barrier(0);
        fold(acc[0], q[0]);
        st = st_next;
        continue;
      }
      auto tile = [&](auto tile_c) {
        constexpr int i = decltype(tile_c)::value, p = i & 1, prev = i == RT - 1 ? 0 : i + 1;
        // the fragments that take this tile's registers: two tiles on in this block, or of the next one's first two
        constexpr int f = i > 1 ? i - 2 : (T1 & 1) == p ? T1 : T2;
        if constexpr (BLK) q[qi(i)] = mm_half(wf[0], x[p][0], zero16);
        else acc[i] = mm_half(wf[0], x[p][0], acc[i]);
        __builtin_amdgcn_sched_group_barrier(0x8, MPH, 0);
        if constexpr (i == 1) {
          if constexpr (BLK) q[qi(i)] = mm_half(wf[1], x[p][1], q[qi(i)]);
          else acc[i] = mm_half(wf[1], x[p][1], acc[i]);
          __builtin_amdgcn_sched_group_barrier(0x8, MPH, 0);
          __builtin_amdgcn_sched_barrier(0);
          // every fragment of this block is in registers; behind the barrier the next block is in LDS
          asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
          __builtin_amdgcn_s_barrier();
          asm volatile("" : "+v"(x[0][0]), "+v"(x[0][1]) : : "memory");
          __builtin_amdgcn_sched_barrier(0);
          x[p][0] = frag(then + A_OFF + f * 4096, 0);
          x[p][1] = frag(then + A_OFF + f * 4096, 1);
          if constexpr (BLK) {
            const bool last = kb + 1 == nkb;
            sbv_n = *(last ? sb0_next : sb0 + kb + 1);
            sbv1_n = *(last ? sb1_next : sb1 + kb + 1);
          }
          fold(acc[prev], q[qi(prev)]);
        } else {
          if constexpr (i == 0) wf[0] = frag(then + wave * 4096, 0);
          x[p][0] = frag((i > 1 ? now : then) + A_OFF + f * 4096, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, i == 0 ? 4 : 2, 0);
          fold(acc[prev], q[qi(prev)]);
          if constexpr (BLK) __builtin_amdgcn_sched_group_barrier(0x2, FOLDN, 0);
          if constexpr (BLK) q[qi(i)] = mm_half(wf[1], x[p][1], q[qi(i)]);
          else acc[i] = mm_half(wf[1], x[p][1], acc[i]);
          __builtin_amdgcn_sched_group_barrier(0x8, MPH, 0);
          if constexpr (i == 0) wf[1] = frag(then + wave * 4096, 1);
          x[p][1] = frag((i > 1 ? now : then) + A_OFF + f * 4096, 1);
        }
        if constexpr (BLK) {
          sc = sa[p] * sbv;
          sc1 = sa[p] * sbv1;
          sa[p] = row_scale(i > 1 ? now : then, f);
        }
        __builtin_amdgcn_sched_barrier(0);
      };
      if constexpr (RT > 3) tile(std::integral_constant<int, 3>{});
      if constexpr (RT > 2) tile(std::integral_constant<int, 2>{});
      if constexpr (RT > 1) {
        tile(std::integral_constant<int, 1>{});
        tile(std::integral_constant<int, 0>{});
      }
      sbv = sbv_n;
      sbv1 = sbv1_n;
      st = st_next;
    }
    if constexpr (RT > 1) fold(acc[0], q[0]);

    // ---- the finished tile leaves; the next one's first blocks are on their way -----------------------------------
    const int n0 = pn * R, n_end = min(n0 + R, (int)g.N), nw = n0 + wave * 32;
    if (slices > 1) {
      float* slab = (float*)g.C + (int64_t)slice * g.M * g.N;
#pragma unroll
      for (int i = 0; i < RT; i++) {
        const int m = i * 32 + frow;
        if (m >= g.M) continue;
#pragma unroll
        for (int rq = 0; rq < 4; rq++) {
          const int n = nw + 8 * rq + 4 * fk;
          if (n >= n_end) continue;
          float v[4];
#pragma unroll
          for (int r = 0; r < 4; r++) {
            if constexpr (MODE == GEMM_ROW_INT8) v[r] = __int_as_float(acc[i][rq * 4 + r]);
            else v[r] = acc[i][rq * 4 + r];
          }
          float* prow = slab + (int64_t)m * g.N + n;
          if (n + 3 < n_end && ((((uintptr_t)prow) & 15) == 0)) {
            *(v4f*)prow = v4f{v[0], v[1], v[2], v[3]};
          } else {
            for (int r = 0; r < 4 && n + r < n_end; r++) prow[r] = v[r];
          }
        }
      }
    } else {
      // wave-private staging: 32 rows of 64 bytes, 16-byte pieces swizzled with the row
      uint8_t* stg = smem + PATCH_BASE + wave * 2048;
      float sbn[16], bia[16];
      if constexpr (!BLK) {
#pragma unroll
        for (int r = 0; r < 16; r++) {
          const int nn = min(nw + 8 * (r >> 2) + 4 * fk + (r & 3), (int)g.N - 1);
          sbn[r] = g.sb[nn];
          bia[r] = g.bias ? OT::to_f32(((const OS*)g.bias)[nn]) : 0.f;
        }
      }
      const int piece = lane & 3, n = nw + piece * 8;
      v4i bias8 = {};
      if constexpr (out_biased<OT>) {
        OS b[8];
#pragma unroll
        for (int r = 0; r < 8; r++) b[r] = ((const OS*)g.bias)[min(n + r, (int)g.N - 1)];
        __builtin_memcpy(&bias8, b, 16);
      }
#pragma unroll
      for (int i = 0; i < RT; i++) {
        float sam = 1.f;
        if constexpr (!BLK) sam = g.sa[min(i * 32 + frow, (int)g.M - 1)];
        float v[16];
#pragma unroll
        for (int r = 0; r < 16; r++) {
          v[r] = (float)acc[i][r];
          if constexpr (!BLK) {
            if constexpr (MODE == GEMM_ROW_FP8) v[r] = v[r] * sbn[r] * sam;
            else v[r] = v[r] * (sbn[r] * sam);
            if (g.bias) v[r] += bia[r];
          }
        }
#pragma unroll
        for (int rq = 0; rq < 4; rq++) {
          const v2i w = {(int)OT::pack2(v[rq * 4], v[rq * 4 + 1]), (int)OT::pack2(v[rq * 4 + 2], v[rq * 4 + 3])};
          *(v2i*)(stg + frow * 64 + ((rq ^ ((frow >> 2) & 3)) << 4) + fk * 8) = w;
        }
#pragma unroll
        for (int half = 0; half < 2; half++) {
          const int row = (lane >> 2) + 16 * half;
          v4i o = *(const v4i*)(stg + row * 64 + ((piece ^ ((row >> 2) & 3)) << 4));
          if constexpr (out_biased<OT>) o = add_bias8<OT>(o, bias8);
          const int m = i * 32 + row;
          if (m >= g.M || n >= n_end) continue;
          OS* dst = (OS*)g.C + (int64_t)m * g.ldc + n;
          if (n + 8 <= n_end && ((((uintptr_t)dst) & 15) == 0)) {
            *(v4i*)dst = o;
          } else {
            OS e[8];
            __builtin_memcpy(e, &o, 16);
            for (int r = 0; r < 8 && n + r < n_end; r++) dst[r] = e[r];
          }
        }
      }
    }
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][r] = 0;
#pragma unroll
    for (int r = 0; r < 16; r++) q[0][r] = 0;
    sc = sc1 = 0.f;
    sb0 = sb0_next;
    sb1 = sb1_next;
    buf ^= 1;
  }
#endif
}

struct StripPlan {
  int rows = 0, slices = 1;  // weight rows of a tile, K slices
  double us = 1e30;
};
// Strips of 32 weight rows, and stages in LDS, of the kernel that runs tiles of `rows` weight rows.
static inline int strip_strips(int64_t M, int rows) { return rows <= 96 && M <= 32 ? 3 : rows <= 128 ? 4 : 5; }
static inline int strip_depth(int64_t M, int rows) {
  const int ns = strip_strips(M, rows);
  return M > 32 ? strip_stages<2, 4>() : ns == 3 ? strip_stages<1, 3>() : ns == 4 ? strip_stages<1, 4>() : strip_stages<1, 5>();
}
// The weight scales of the block modes lie in two tables, those of an item and of the one behind it.  The loading waves
// write the table of item j + 2 over that of item j as soon as the request stream, as many blocks ahead of the products as
// there are stages, enters it: item j's last block has passed its barrier by then if item j + 1 has at least stages - 1 blocks.
// With fewer (17 x 790016 x 128: one block an item, five stages) a workgroup may only have two items.
static inline bool strip_tables_hold(int64_t M, int64_t N, int64_t K, const StripPlan& plan) {
  const int64_t items = ceil_div(N, plan.rows) * plan.slices;
  return items <= 2 * (int64_t)device_cus() || (K >> 7) / plan.slices >= strip_depth(M, plan.rows) - 1;
}
// What the kernel takes: 32-bit offsets, whole K blocks in the block modes and enough of them for the scale tables.
template <int MODE>
static inline bool strip_ok(const GemmArgs& g, const StripPlan& plan) {
  if (g.M < 17 || g.M > STRIP_MAX_ROWS || !gemm8_big_ok(g, !gemm_is_block(MODE))) return false;
  if (!gemm_is_block(MODE)) return true;
  const int64_t nkb = g.K >> 7;
  return strip_tables_hold(g.M, g.N, g.K, plan) && ((int64_t)(g.M - 1) * g.sa_sm + (nkb - 1) * g.sa_sk + 1) * 4 < 0x7ffffff0ll &&
         ((nkb - 1) * g.sb_sk + 1) * 4 < 0x7ffffff0ll;
}

// The tile and the number of K slices of a launch, and its time in us without what all forms have in common (launch, quantiser):
// rounds of items x (K blocks of an item x the time of a block + its drain), and a second launch where K is split.  A
// block takes the longer of the multiplying wave's chain and the bytes' way in, and half of the other.  Fitted to 4752 launches
// of 92 weights of 0.3 to 470 MB, three scaling modes, weights from HBM and from the Infinity Cache: 7 % rms.
static inline StripPlan strip_plan(int64_t M, int64_t N, int64_t K) {
  StripPlan best;
  const int64_t nkb = (K + 127) >> 7, cus = device_cus();
  const int rt = M <= 32 ? 1 : M <= 64 ? 2 : M <= 96 ? 3 : 4;
  const double chain = rt == 1 ? 0.13 : rt == 2 ? 0.247 : rt == 3 ? 0.366 : 0.470;
  for (int rows = 32; rows <= 160; rows += 16) {
    const int64_t tiles = (N + rows - 1) / rows;
    for (int slices = 1; slices <= 12; slices++) {
      if (slices > 1 && ((N & 3) || nkb / slices < 4)) break;
      if (nkb > (int64_t)slices * STRIP_MAX_KB) continue;
      const int64_t items = tiles * slices, rounds = (items + cus - 1) / cus;
      const double fill = items < cus ? (double)items / cus : 1.0;
      const double own = chain * (rows > 128 ? 1.36 : 1.0), in = ((rt == 1 ? 0.0040 : 0.0032) * rows + 0.016 * rt) * fill * (1.2 - 0.2 * fill);
      double us = rounds * ((double)nkb / slices * (own > in ? own + 0.47 * in : in + 0.47 * own) + 2.85);
      // (as many items as CUs and short ones: all of them write their slabs at once, 10 to 18 % on top at 96 rows and more)
      if (slices > 1) us = us * (items == cus && nkb < 32 * slices && M > 64 ? 1.1 : 1.0) + 3.2 + (double)slices * M * N * 1.48e-6;
      if (us < best.us) best.rows = rows, best.slices = slices, best.us = us;
    }
  }
  return best;
}

template <int MODE, typename OT, int RT, int NS>
static int gemm8_strip_start(const GemmArgs& g, hipStream_t st) {
  auto kern = gemm8_strip_kernel<MODE, OT, RT, NS>;
  constexpr int smem = strip_smem<MODE, RT, NS>();
  static_assert(smem <= 160 * 1024, "LDS of a CU");
  static SmemAttrOnce attr;
  hipError_t e = raise_dynamic_smem(attr, (const void*)kern, smem);
  if (e != hipSuccess) return fail(SGLAMD_EHIP, "hipFuncSetAttribute: %s", hipGetErrorString(e));
  const int64_t items = ceil_div(g.N, g.rows_per_wg) * g.max_blocks_m;
  hipLaunchKernelGGL(kern, dim3((unsigned)(items < device_cus() ? items : device_cus())), dim3(512), smem, st, g);
  return check_launch("gemm8_strip");
}
// `workspace`: plan.slices * M * N fp32 where K is split.
template <int MODE, typename OT>
static int gemm8_strip_launch(const GemmArgs& whole, const StripPlan& plan, hipStream_t st, void* workspace) {
  GemmArgs g = whole;
  g.rows_per_wg = plan.rows;
  g.max_blocks_m = plan.slices;
  // Weights that the 256 MB Infinity Cache cannot keep beside everything else are read past the caches: 36864 x 7168 at 64 rows 49.5
  // -> 44 us.  Smaller ones may come from there.
  g.streams = (int64_t)g.N * g.K >= (96ll << 20);
  if (plan.slices > 1) g.C = workspace;
  int rc;
  auto start = [&](auto ns) {
    constexpr int NS = decltype(ns)::value;
    if (g.M <= 32) return gemm8_strip_start<MODE, OT, 1, NS>(g, st);
    if constexpr (NS == 3) return gemm8_strip_start<MODE, OT, 2, 4>(g, st);
    else return g.M <= 64 ? gemm8_strip_start<MODE, OT, 2, NS>(g, st) : g.M <= 96 ? gemm8_strip_start<MODE, OT, 3, NS>(g, st) : gemm8_strip_start<MODE, OT, 4, NS>(g, st);
  };
  const int ns = strip_strips(g.M, plan.rows);
  if (ns == 3) rc = start(std::integral_constant<int, 3>{});
  else if (ns == 4) rc = start(std::integral_constant<int, 4>{});
  else rc = start(std::integral_constant<int, 5>{});
  if (rc || plan.slices == 1) return rc;
  return splitk_reduce<MODE, OT>(whole, plan.slices, workspace, st);
}

}  // namespace sglamd
