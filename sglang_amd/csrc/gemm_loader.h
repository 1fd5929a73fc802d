#pragma once
#include "gemm_big.h"

namespace sglamd {

constexpr int LOADER_STAGES = 3;
constexpr int LOADER_MAX_KB = 256;
template <int MODE>
constexpr int loader_stage() {
  return (256 + 128) * 128 + (gemm_is_block(MODE) ? 512 : 0);
}
template <int MODE>
constexpr int loader_smem() {
  return LOADER_STAGES * loader_stage<MODE>() + 4 * 2048 + (gemm_is_block(MODE) ? 2 * 2 * LOADER_MAX_KB * 4 : 0);
}

template <int MODE, typename OT>
__global__ __launch_bounds__(512) void gemm8_loader_kernel(GemmArgs g) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr bool BLK = gemm_is_block(MODE);
  constexpr int RT = 4, NS = 4, BM = 32 * RT, BN = 64 * NS, D = LOADER_STAGES, NL = 4;
  // wave-wide loads of a K block: groups of eight weight rows, of eight rows, of 64 row scales; loading wave l issues l, l + NL, ...
  constexpr int WG = BN / 8, AG = BM / 8, SG = BLK ? BM / 64 : 0, UNITS = WG + AG + SG;
  constexpr int LPB = (UNITS + NL - 1) / NL;
  constexpr int STAGE = loader_stage<MODE>(), A_OFF = WG * 1024, S_OFF = A_OFF + AG * 1024;
  constexpr int PATCH_BASE = D * STAGE, TBL_BASE = PATCH_BASE + NS * 2048, TBL_BYTES = 2 * LOADER_MAX_KB * 4;
  static_assert((D - 1) * LPB < 64, "vmcnt field is 6 bits");
  typedef typename std::conditional<MODE == GEMM_ROW_INT8, v16i, v16f>::type acc16_t;
  typedef typename std::conditional<gemm_is_int8(MODE), v16i, v16f>::type prod16_t;
  typedef typename OT::storage OS;
  static_assert(sizeof(OS) == 2, "2-byte outputs");

  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  const int slices = g.max_blocks_m;
  const int tiles_m = (g.M + BM - 1) / BM, tiles_n = (g.N + BN - 1) / BN, tiles = tiles_m * tiles_n, items = tiles * slices;
  const int G = (int)gridDim.x;
  const int nkb_all = g.K >> 7;
  // item: slice by slice; in a slice groups of eight row tiles share their weight columns back to back
  struct Item {
    int m0, n0, slice, kb, nkb;
  };
  auto item_at = [&](int p) -> Item {
    const int slice = __builtin_amdgcn_readfirstlane(p / tiles), t = p - slice * tiles;
    const int group = __builtin_amdgcn_readfirstlane(t / (8 * tiles_n)), in = t - group * 8 * tiles_n;
    const int rows = min(tiles_m - group * 8, 8), col = __builtin_amdgcn_readfirstlane(in / rows);
    const int kb = __builtin_amdgcn_readfirstlane(nkb_all * slice / slices), end = __builtin_amdgcn_readfirstlane(nkb_all * (slice + 1) / slices);
    return Item{(group * 8 + in - col * rows) * BM, col * BN, slice, kb, end - kb};
  };
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
    auto dma4 = [&](const v4i& rs, uint32_t voff, int soff, uint32_t lds_off) {
      asm volatile("s_nop 4\n\tbuffer_load_dword %0, %1, %2 offen lds" : : "v"(voff), "s"(rs), "s"(soff), "{m0}"(smem_base + lds_off) : "memory");
    };
    const v4i a_rs = descriptor(g.A, (int64_t)g.M * g.lda), b_rs = descriptor(g.B, (int64_t)g.N * g.ldb);
    const v4i s_rs = descriptor(g.sa, BLK ? ((int64_t)(g.M - 1) * g.sa_sm + (int64_t)(nkb_all - 1) * g.sa_sk + 1) * 4 : 0);

    // the request stream: block `rk` of item `at`
    uint32_t voff[LPB];
    int at = first, rk = 0, r_nkb = 0, r_begin = 0, r_stage = 0, r_buf = 0;
    auto enter = [&]() {
      const Item it = item_at(at);
      r_begin = it.kb;
      r_nkb = it.nkb;
      rk = 0;
#pragma unroll
      for (int u = 0; u < LPB; u++) {
        const int e = u * NL + loader;
        const int row = (e < WG ? e : e - WG) * 8 + (lane >> 3), chunk = (lane & 7) ^ ((row >> 1) & 7);
        const int srow = min(it.m0 + max(e - WG - AG, 0) * 64 + lane, (int)g.M - 1);
        if (e < WG) voff[u] = it.n0 + row < g.N ? (uint32_t)((it.n0 + row) * (int)g.ldb + chunk * 16) : OUTSIDE;
        else if (e < WG + AG) voff[u] = it.m0 + row < g.M ? (uint32_t)((it.m0 + row) * (int)g.lda + chunk * 16) : OUTSIDE;
        else voff[u] = (uint32_t)(srow * (int)g.sa_sm) << 2;
      }
      if constexpr (BLK) {
        // weight scales of the tile's two column blocks
        const int chunks = (r_nkb + 63) >> 6;
        const int64_t span = ((int64_t)(nkb_all - 1) * g.sb_sk + 1) * 4;
        for (int c = loader; c < 2 * chunks; c += NL) {
          const int cb = c >= chunks, kb = (c - cb * chunks) * 64 + lane;
          const int row = __builtin_amdgcn_readfirstlane(min(it.n0 + cb * 128, (int)g.N - 1) >> 7);
          dma4(descriptor(g.sb + (int64_t)row * g.sb_sn, span), kb < r_nkb ? (uint32_t)((r_begin + kb) * (int)g.sb_sk) << 2 : OUTSIDE, 0,
               __builtin_amdgcn_readfirstlane(TBL_BASE + r_buf * TBL_BYTES + (cb * LOADER_MAX_KB + (c - cb * chunks) * 64) * 4));
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
      const int kq = __builtin_amdgcn_readfirstlane(rk + r_begin);
      const int stage = __builtin_amdgcn_readfirstlane(r_stage * STAGE);
#pragma unroll
      for (int u = 0; u < LPB; u++) {
        const int e = u * NL + loader;
        const uint32_t to = (uint32_t)(stage + e * 1024);
        if (u * NL + NL <= WG || e < WG) {
          dma16(b_rs, voff[u], kq << 7, to);
        } else if (u * NL + NL <= WG + AG || e < WG + AG) {
          dma16(a_rs, voff[u], kq << 7, to);
        } else if (u * NL + NL <= UNITS || e < UNITS) {
          dma4(s_rs, voff[u], (kq * (int)g.sa_sk) << 2, (uint32_t)(stage + S_OFF + (e - WG - AG) * 256));
        }
      }
      rk++;
      r_stage = r_stage == D - 1 ? 0 : r_stage + 1;
    };
    const bool full = UNITS % NL == 0 || (LPB - 1) * NL + loader < UNITS;  // issues LPB loads a block, not one less
    // all but the last `blocks` blocks requested have landed
#define STRIP_LANDED(blocks)                                                          \
  if (full) asm volatile("s_waitcnt vmcnt(%0)" : : "n"((blocks)*LPB) : "memory");     \
  else asm volatile("s_waitcnt vmcnt(%0)" : : "n"((blocks) * (LPB - 1)) : "memory")
    int left = 0;  // blocks of this workgroup's items
    for (int it = first; it < items; it += G) {
      left += item_at(it).nkb;
    }
    enter();
    for (int d = 0; d < D; d++) request();
    if (left >= D) {
      STRIP_LANDED(D - 1);
    } else {
      asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
    }
    __builtin_amdgcn_s_barrier();
    for (; left > 0; left--) {
      // the next block has landed; behind the barrier this one is in the multiplying waves' registers, and its stage is free
      if (left >= D) {
        STRIP_LANDED(D - 2);
      } else {
        asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
      }
      __builtin_amdgcn_s_barrier();
      request();
    }
#undef STRIP_LANDED
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
  acc16_t acc[RT][2];
  prod16_t qa, qb, zero16;  // products of a row tile with the wave's two column tiles; qb waits for the next tile's
#pragma unroll
  for (int i = 0; i < RT; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][j][r] = 0;
#pragma unroll
  for (int r = 0; r < 16; r++) qa[r] = 0, qb[r] = 0, zero16[r] = 0;
  float scp = 0.f;
  // half of a product's sixteen values
  auto fold = [&](acc16_t& dst, const prod16_t& p, int half) {
    if constexpr (BLK) {
#pragma unroll
      for (int r = 0; r < 8; r++) dst[half * 8 + r] = fmaf((float)p[half * 8 + r], scp, dst[half * 8 + r]);
    }
  };
  auto row_scale = [&](int stage, int t) -> float { return *(const float*)(smem + stage + S_OFF + (t * 32 + frow) * 4); };

  __builtin_amdgcn_s_barrier();  // block 0 has landed
  asm volatile("" : : : "memory");
  int st = 0, buf = 0;
  for (int item = first; item < items; item += G) {
    const Item it = item_at(item);
    const int nkb = it.nkb;
    const float* sb = (const float*)(smem + TBL_BASE + buf * TBL_BYTES) + (wave >> 1) * LOADER_MAX_KB;
    // the first block has landed (the barrier of the block in front of it)
    v8i wf[2][2], x[2][2];  // [column tile][K half], [parity of the row tile][K half]
    float sa[2] = {1.f, 1.f}, sbv = 1.f;
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int h = 0; h < 2; h++) {
        wf[j][h] = frag(st * STAGE + wave * 8192 + j * 4096, h);
        x[j][h] = frag(st * STAGE + A_OFF + j * 4096, h);
      }
    if constexpr (BLK) sa[0] = row_scale(st * STAGE, 0), sa[1] = row_scale(st * STAGE, 1), sbv = sb[0];

    for (int kb = 0; kb < nkb; kb++) {
      const int now = st * STAGE, st_next = st == D - 1 ? 0 : st + 1, then = st_next * STAGE;
      float sbv_n = 1.f;
      // Each product is followed by what issues in its shadow, some fifteen instructions: fragment and scale reads, then half
      // of a fold, which so lies the eighteen issue slots behind the product that it needs.
      auto tile = [&](auto tile_c) {
        constexpr int i = decltype(tile_c)::value, p = i & 1, prev = i == 0 ? RT - 1 : i - 1;
        constexpr int f = (i + 2) & (RT - 1);  // the row tile whose fragments take this one's registers
        constexpr bool last = i == RT - 1;
        const int from = (i < RT - 2 ? now : then) + A_OFF + f * 4096;
#define SLOT __builtin_amdgcn_sched_barrier(0)
        if constexpr (BLK) qa = mm_half(wf[0][0], x[p][0], zero16);
        else acc[i][0] = mm_half(wf[0][0], x[p][0], acc[i][0]);
        SLOT;
        if constexpr (last) wf[0][0] = frag(then + wave * 8192, 0);
        SLOT;
        fold(acc[prev][1], qb, 0);
        SLOT;
        if constexpr (BLK) qa = mm_half(wf[0][1], x[p][1], qa);
        else acc[i][0] = mm_half(wf[0][1], x[p][1], acc[i][0]);
        SLOT;
        if constexpr (last) wf[0][1] = frag(then + wave * 8192, 1);
        SLOT;
        fold(acc[prev][1], qb, 1);
        if constexpr (BLK) scp = sa[p] * sbv;
        if constexpr (i == RT - 2) {
          // every fragment of this block is in registers; behind the barrier the next block is in LDS
          asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
          __builtin_amdgcn_s_barrier();
          asm volatile("" : "+v"(x[p][0]), "+v"(x[p][1]) : : "memory");
        }
        SLOT;
        if constexpr (BLK) qb = mm_half(wf[1][0], x[p][0], zero16);
        else acc[i][1] = mm_half(wf[1][0], x[p][0], acc[i][1]);
        SLOT;
        x[p][0] = frag(from, 0);
        if constexpr (last) wf[1][0] = frag(then + wave * 8192 + 4096, 0);
        if constexpr (BLK) sa[p] = row_scale(i < RT - 2 ? now : then, f);
        if constexpr (BLK && i == RT - 2) sbv_n = sb[min(kb + 1, nkb - 1)];
        SLOT;
        fold(acc[i][0], qa, 0);
        SLOT;
        if constexpr (BLK) qb = mm_half(wf[1][1], x[p][1], qb);
        else acc[i][1] = mm_half(wf[1][1], x[p][1], acc[i][1]);
        SLOT;
        x[p][1] = frag(from, 1);
        if constexpr (last) wf[1][1] = frag(then + wave * 8192 + 4096, 1);
        SLOT;
        fold(acc[i][0], qa, 1);
        SLOT;
#undef SLOT
      };
      tile(std::integral_constant<int, 0>{});
      tile(std::integral_constant<int, 1>{});
      tile(std::integral_constant<int, 2>{});
      tile(std::integral_constant<int, 3>{});
      sbv = sbv_n;
      st = st_next;
    }
    fold(acc[RT - 1][1], qb, 0);
    fold(acc[RT - 1][1], qb, 1);

    // ---- the finished tile leaves; the next one's first blocks are on their way -----------------------------------
    int ln = lane;
    asm volatile("" : "+v"(ln));  // (the output's lane arithmetic would live in registers through the K loop)
    const int orow = ln & 31, ok = ln >> 5;
    const int m0 = it.m0, nw = it.n0 + wave * 64;
    if (slices > 1) {
      float* slab = (float*)g.C + (int64_t)it.slice * g.M * g.N;
#pragma unroll
      for (int i = 0; i < RT; i++) {
        const int m = m0 + i * 32 + orow;
        if (m >= g.M) continue;
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
          for (int rq = 0; rq < 4; rq++) {
            const int n = nw + j * 32 + 8 * rq + 4 * ok;
            if (n >= g.N) continue;
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
              if constexpr (MODE == GEMM_ROW_INT8) v[r] = __int_as_float(acc[i][j][rq * 4 + r]);
              else v[r] = acc[i][j][rq * 4 + r];
            }
            float* prow = slab + (int64_t)m * g.N + n;
            if (n + 3 < g.N && ((((uintptr_t)prow) & 15) == 0)) {
              *(v4f*)prow = v4f{v[0], v[1], v[2], v[3]};
            } else {
              for (int r = 0; r < 4 && n + r < g.N; r++) prow[r] = v[r];
            }
          }
      }
    } else {
      // wave-private staging: 32 rows of 64 bytes, 16-byte pieces swizzled with the row
      uint8_t* stg = smem + PATCH_BASE + wave * 2048;
      const int piece = ln & 3;
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const int nj = nw + j * 32, n = nj + piece * 8;
        float sbn[16], bia[16];
        if constexpr (!BLK) {
#pragma unroll
          for (int r = 0; r < 16; r++) {
            const int nn = min(nj + 8 * (r >> 2) + 4 * ok + (r & 3), (int)g.N - 1);
            sbn[r] = g.sb[nn];
            bia[r] = g.bias ? OT::to_f32(((const OS*)g.bias)[nn]) : 0.f;
          }
        }
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
          if constexpr (!BLK) sam = g.sa[min(m0 + i * 32 + orow, (int)g.M - 1)];
          float v[16];
#pragma unroll
          for (int r = 0; r < 16; r++) {
            v[r] = (float)acc[i][j][r];
            if constexpr (!BLK) {
              if constexpr (MODE == GEMM_ROW_FP8) v[r] = v[r] * sbn[r] * sam;
              else v[r] = v[r] * (sbn[r] * sam);
              if (g.bias) v[r] += bia[r];
            }
          }
#pragma unroll
          for (int rq = 0; rq < 4; rq++) {
            const v2i w = {(int)OT::pack2(v[rq * 4], v[rq * 4 + 1]), (int)OT::pack2(v[rq * 4 + 2], v[rq * 4 + 3])};
            *(v2i*)(stg + orow * 64 + ((rq ^ ((orow >> 2) & 3)) << 4) + ok * 8) = w;
          }
#pragma unroll
          for (int half = 0; half < 2; half++) {
            const int row = (ln >> 2) + 16 * half;
            v4i o = *(const v4i*)(stg + row * 64 + ((piece ^ ((row >> 2) & 3)) << 4));
            if constexpr (out_biased<OT>) o = add_bias8<OT>(o, bias8);
            const int m = m0 + i * 32 + row;
            if (m >= g.M || n >= g.N) continue;
            OS* dst = (OS*)g.C + (int64_t)m * g.ldc + n;
            if (n + 8 <= g.N && ((((uintptr_t)dst) & 15) == 0)) {
              *(v4i*)dst = o;
            } else {
              OS e[8];
              __builtin_memcpy(e, &o, 16);
              for (int r = 0; r < 8 && n + r < g.N; r++) dst[r] = e[r];
            }
          }
        }
      }
    }
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
      for (int j = 0; j < 2; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[i][j][r] = 0;
#pragma unroll
    for (int r = 0; r < 16; r++) qb[r] = 0;
    scp = 0.f;
    buf ^= 1;
  }
#endif
}

}  // namespace sglamd
