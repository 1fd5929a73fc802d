// Per-token-group quantisation body shared by the stand-alone quant kernels and the fused-MoE
// prologue kernel (which quantises the hidden states in the same launch that sorts the tokens).
#pragma once
#include "common.h"

namespace sglamd {

// ceil(log2(x)) for a positive normal float, from its bit pattern.
__device__ __forceinline__ int log2_ceil_bits(float x) {
  uint32_t b = __float_as_uint(x);
  int e = (int)((b >> 23) & 0xff);
  return e - 127 + ((b & 0x7fffffu) != 0);
}
__device__ __forceinline__ float pow2_int(int e) { return __uint_as_float((uint32_t)(e + 127) << 23); }

template <int WIDTH>
__device__ __forceinline__ float group_max(float v) {
#pragma unroll
  for (int off = WIDTH / 2; off >= 1; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  return v;
}

struct GroupQuantArgs {
  const void* in;
  void* q;
  void* s;
  int64_t num_groups;      // rows * groups_per_row
  int groups_per_row;
  FastDiv per_row;         // division by groups_per_row; used while num_groups < 2^31
  int layout;
  int64_t scale_stride;    // column-major: between groups; PITCHED row-major: floats from row to row
  float eps, min8, max8;
  int form;
  int q_is_fp8;
  int pow2;                // scales rounded up to powers of two (implied by the UE8M0 layout)
  int64_t hidden;          // output elements per row
  // masked (DeepEP) layout: rows are [expert][token]; only tokens < masked_m[expert] are quantised, and the
  // UE8M0 scale words of expert e start scale_expert_stride int32 words after those of expert e-1
  const int32_t* masked_m;
  int tokens_per_expert;
  int64_t scale_expert_stride;

  void set_rows(int64_t rows, int64_t hidden_, int group) {
    hidden = hidden_;
    groups_per_row = (int)(hidden_ / group);
    num_groups = rows * groups_per_row;
    per_row = FastDiv::of((uint32_t)groups_per_row);
  }
};

// T: input storage tag; GROUP: elements per group.  ELEMS elements per lane (32 bytes),
// LPG = GROUP / ELEMS lanes share a group.  SILU: input rows are [gate | up] of 2 * hidden and
// x = T(silu(gate)) * up rounded to T.  PITCHED: rows of row-major scales lie scale_stride floats apart.
//
// HBM-bound as long as its instructions stay few: a wave64 VALU instruction takes a SIMD four cycles, so a lane's 16
// elements may cost about 350 instructions before the arithmetic is the slower side.  Hence no 64-bit divisions, the
// clamp as one v_med3_f32 (NaN in, lower bound out, like fmin(fmax())), and silu_rounded.  8192 bf16 rows of
// 18432 gates and 18432 ups, UE8M0 scales: 170 -> 133 us (5.7 TB/s; a plain copy moves 5.1); of 7168 and 7168: 67 -> 51.
template <typename T, int GROUP, bool SILU = false, bool PITCHED = false>
__device__ __forceinline__ void group_quant_body(const GroupQuantArgs& a, const int64_t lane_global) {
  typedef typename T::storage S;
  constexpr int ELEMS = 32 / (int)sizeof(S);
  constexpr int LPG = GROUP / ELEMS;
  static_assert(LPG >= 1 && LPG <= 64 && (LPG & (LPG - 1)) == 0, "group must span 1..64 lanes");

  const int64_t g = lane_global / LPG;
  const int sub = (int)(lane_global % LPG);
  bool active = g < a.num_groups;
  const bool row_major = a.layout == SGLAMD_SCALE_ROW_MAJOR;
  // row and group inside the row, where something below needs them
  auto locate = [&](int64_t gg, int64_t& row, int& col) {
    if (a.num_groups <= 0x7fffffff) {
      const uint32_t r = a.per_row.divide((uint32_t)gg);
      row = r;
      col = (int)((uint32_t)gg - r * (uint32_t)a.groups_per_row);
    } else {
      row = gg / a.groups_per_row;
      col = (int)(gg % a.groups_per_row);
    }
  };
  int64_t row = 0;
  int col = 0;
  if (SILU && a.masked_m && active) {
    locate(g, row, col);
    active = (int)((uint32_t)row % (uint32_t)a.tokens_per_expert) < a.masked_m[(uint32_t)row / (uint32_t)a.tokens_per_expert];
  }
  // Lanes past the end keep running (they take part in the cross-lane max) on group 0's
  // address range but store nothing.
  const int64_t gg = active ? g : 0;
  if (SILU || !row_major || PITCHED) locate(gg, row, col);

  float x[ELEMS];
  float amax = a.eps;
  if constexpr (!SILU) {
    const S* src = (const S*)a.in + gg * GROUP + sub * ELEMS;
    v4i raw0 = *(const v4i*)src;
    v4i raw1 = *((const v4i*)src + 1);
    S buf[ELEMS];
    __builtin_memcpy(&buf[0], &raw0, 16);
    __builtin_memcpy(&buf[ELEMS / 2], &raw1, 16);
#pragma unroll
    for (int i = 0; i < ELEMS; i++) x[i] = T::to_f32(buf[i]);
  } else {
    // gate and up halves of one [2*hidden] row; silu is rounded to T, the product is rounded to T
    const S* gsrc = (const S*)a.in + row * 2 * a.hidden + (int64_t)col * GROUP + sub * ELEMS;
    const S* usrc = gsrc + a.hidden;
    v4i g0 = *(const v4i*)gsrc, g1 = *((const v4i*)gsrc + 1);
    v4i u0 = *(const v4i*)usrc, u1 = *((const v4i*)usrc + 1);
    S gb[ELEMS], ub[ELEMS];
    __builtin_memcpy(&gb[0], &g0, 16);
    __builtin_memcpy(&gb[ELEMS / 2], &g1, 16);
    __builtin_memcpy(&ub[0], &u0, 16);
    __builtin_memcpy(&ub[ELEMS / 2], &u1, 16);
#pragma unroll
    for (int i = 0; i < ELEMS; i++)
      x[i] = T::to_f32(T::from_f32(silu_rounded<T>(T::to_f32(gb[i])) * T::to_f32(ub[i])));
  }
#pragma unroll
  for (int i = 0; i < ELEMS; i++) amax = fmaxf(amax, fabsf(x[i]));
  amax = group_max<LPG>(amax);

  const bool ue8m0 = a.layout == SGLAMD_SCALE_COL_MAJOR_UE8M0;
  const bool pow2 = ue8m0 || a.pow2;
  float s_store;   // value written as the scale (or whose exponent byte is written)
  float mul = 0.f; // reciprocal form: multiplier applied to x
  if (a.form == SGLAMD_QUANT_FORM_DIVIDE) {
    s_store = amax / a.max8;
    if (pow2) s_store = pow2_int(log2_ceil_bits(fmaxf(s_store, 1e-10f)));
  } else {
    if (pow2) {
      int e = log2_ceil_bits(amax * (1.0f / a.max8));
      mul = pow2_int(-e);
      s_store = pow2_int(e);
    } else {
      s_store = amax * (1.0f / a.max8);
      mul = a.max8 / amax;
    }
  }

  float y[ELEMS];
  if (a.form == SGLAMD_QUANT_FORM_DIVIDE) {
#pragma unroll
    for (int i = 0; i < ELEMS; i++) y[i] = __builtin_amdgcn_fmed3f(x[i] / s_store, a.min8, a.max8);
  } else {
#pragma unroll
    for (int i = 0; i < ELEMS; i++) y[i] = __builtin_amdgcn_fmed3f(x[i] * mul, a.min8, a.max8);
  }

  // UE8M0: the four exponent bytes of a word meet in its first group's lanes when the words of a row are whole (then
  // the groups of a word are neighbours of one row); one 4-byte store instead of four single bytes.
  const bool whole_words = GROUP == 128 && LPG == 8 && ue8m0 && (a.groups_per_row & 3) == 0;
  uint32_t word = __float_as_uint(s_store) >> 23;
  if (whole_words) {
    word <<= 8 * (col & 3);
    word |= __shfl_xor(word, 8, 64);
    word |= __shfl_xor(word, 16, 64);
  }
  if (!active) return;

  uint8_t* dst = (uint8_t*)a.q + gg * GROUP + sub * ELEMS;
  uint32_t w[ELEMS / 4];
  if (a.q_is_fp8) {
#pragma unroll
    for (int i = 0; i < ELEMS / 4; i++) w[i] = pack4_e4m3(y[4 * i], y[4 * i + 1], y[4 * i + 2], y[4 * i + 3]);
  } else {
#pragma unroll
    for (int i = 0; i < ELEMS / 4; i++) {
      uint32_t b0 = (uint32_t)(int)y[4 * i] & 0xff, b1 = (uint32_t)(int)y[4 * i + 1] & 0xff;
      uint32_t b2 = (uint32_t)(int)y[4 * i + 2] & 0xff, b3 = (uint32_t)(int)y[4 * i + 3] & 0xff;
      w[i] = b0 | (b1 << 8) | (b2 << 16) | (b3 << 24);
    }
  }
  if constexpr (ELEMS == 16) {
    v4i o = {(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
    *(v4i*)dst = o;
  } else {
    v2i o = {(int)w[0], (int)w[1]};
    *(v2i*)dst = o;
  }

  if (sub == 0) {
    if (row_major) {
      ((float*)a.s)[PITCHED ? row * a.scale_stride + col : gg] = s_store;
    } else if (!ue8m0) {
      ((float*)a.s)[(int64_t)col * a.scale_stride + row] = s_store;
    } else {
      int64_t at = (int64_t)(col >> 2) * a.scale_stride + row;
      if (SILU && a.masked_m) {
        const uint32_t expert = (uint32_t)row / (uint32_t)a.tokens_per_expert;
        at = expert * a.scale_expert_stride + (int64_t)(col >> 2) * a.scale_stride +
             ((uint32_t)row - expert * (uint32_t)a.tokens_per_expert);
      }
      if (whole_words) {
        if ((col & 3) == 0) ((uint32_t*)a.s)[at] = word;
        return;
      }
      uint8_t* sp = (uint8_t*)a.s + (at << 2);
      sp[col & 3] = (uint8_t)word;
      if (col == a.groups_per_row - 1) {
        for (int k = (col & 3) + 1; k < 4; k++) sp[k] = 0;
      }
    }
  }
}

// Per-token (whole row) quantisation of one row by one workgroup of 64 * waves lanes: the row stays in registers
// between the maximum and the conversion (NV pieces of 8 values per lane), so it is read once, all its loads in flight
// together.  SILU: the row is [gate | up] (`up` points at the second half) and what is quantised is
// T(silu(gate)) * up rounded to T, the bytes silu_and_mul would have stored.
// INT8: amax = max(max|x|, 1e-10), s = amax / 127, q = round_half_away(x * (127 / amax));
// FP8:  s = max|x| / 448, q = e4m3(clamp(x * (1 / s))), zeros for a row of zeros.
struct RowQuantArgs {
  const void* in;  // [rows, hidden], SILU: [rows, 2 * hidden]
  void* q;         // [rows, hidden] bytes
  float* s;        // [rows]
  int64_t hidden;  // a multiple of 8
  int64_t rows;
};

// (int)roundf(x) for |x| below 2^22: with the largest float below one half, halves round away from zero and everything under
// them stays (every float up to 200 compared).  Three instructions for roundf's eight: the INT8 rows were bound by their
// arithmetic, 1000 x 28672 values 21.4 -> 18.9 us, 4000 x 18432 52 -> 46.
__device__ __forceinline__ int round_away(float x) {
#pragma clang fp contract(off)  // the scaled value is rounded before the sum
  return (int)(x + copysignf(0x1.fffffep-2f, x));
}
// The low bytes of four integers.
__device__ __forceinline__ uint32_t pack4_low(int a, int b, int c, int d) {
  const uint32_t lo = __builtin_amdgcn_perm((uint32_t)b, (uint32_t)a, 0x0c0c0400u);
  const uint32_t hi = __builtin_amdgcn_perm((uint32_t)d, (uint32_t)c, 0x0c0c0400u);
  return __builtin_amdgcn_perm(hi, lo, 0x05040100u);
}

// TEAM: lanes that share a row, 32 or 64 (no barrier), a multiple of 64, or 0 for the whole workgroup; `row` is the lane's
// own and may be past the end, since every lane takes part in the barrier.
// A row of the experts' activations is 256 to 2048 values: a workgroup per row leaves most of its lanes without work, and
// the launch is bound by starting workgroups (20025 rows of [256 | 256] 34 us, the 25 MB are worth 5).
template <typename T, bool INT8, bool SILU, int NV, int TEAM = 0>
__device__ __forceinline__ void row_quant_body(const RowQuantArgs& a, int64_t row, float* red) {
  typedef typename T::storage S;
  static_assert(sizeof(S) == 2, "16-bit rows");
  const int nt = TEAM ? TEAM : (int)blockDim.x, tid = TEAM ? (int)threadIdx.x % (TEAM ? TEAM : 1) : (int)threadIdx.x;
  const int nvec = row < a.rows ? (int)(a.hidden >> 3) : 0;
  const S* src = (const S*)a.in + row * a.hidden * (SILU ? 2 : 1);
  const S* up = src + a.hidden;
  v4i raw[NV], rup[SILU ? NV : 1];
#pragma unroll
  for (int k = 0; k < NV; k++) {
    const int i = tid + k * nt;
    raw[k] = v4i{0, 0, 0, 0};
    if (SILU) rup[SILU ? k : 0] = v4i{0, 0, 0, 0};
    if (i < nvec) {
      raw[k] = *((const v4i*)src + i);
      if (SILU) rup[SILU ? k : 0] = *((const v4i*)up + i);
    }
  }
  float amax = 0.f;
#pragma unroll
  for (int k = 0; k < NV; k++) {
    S b[8];
    __builtin_memcpy(b, &raw[k], 16);
    if constexpr (SILU) {
      S u[8];
      __builtin_memcpy(u, &rup[k], 16);
#pragma unroll
      for (int j = 0; j < 8; j++) b[j] = T::from_f32(silu_rounded<T>(T::to_f32(b[j])) * T::to_f32(u[j]));
      __builtin_memcpy(&raw[k], b, 16);
    }
#pragma unroll
    for (int j = 0; j < 8; j++) amax = fmaxf(amax, fabsf(T::to_f32(b[j])));
  }
  amax = group_max<TEAM == 32 ? 32 : 64>(amax);
  if constexpr (TEAM != 32 && TEAM != 64) {
    float* mine = red + ((int)threadIdx.x - tid) / 64;
    if ((tid & 63) == 0) mine[tid >> 6] = amax;
    __syncthreads();
    amax = mine[0];
    for (int w = 1; w < (nt >> 6); w++) amax = fmaxf(amax, mine[w]);
  }

  float scale, mul;
  if (INT8) {
    amax = fmaxf(amax, 1e-10f);
    scale = amax / 127.0f;
    mul = 127.0f / amax;
  } else {
    scale = amax / 448.0f;
    mul = (scale == 0.f) ? 0.f : 1.0f / scale;
  }
  if (tid == 0 && row < a.rows) a.s[row] = scale;
  uint8_t* dst = (uint8_t*)a.q + row * a.hidden;
#pragma unroll
  for (int k = 0; k < NV; k++) {
    const int i = tid + k * nt;
    if (i >= nvec) break;
    S b[8];
    __builtin_memcpy(b, &raw[k], 16);
    uint32_t w[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
      float x[4];
#pragma unroll
      for (int j = 0; j < 4; j++) x[j] = T::to_f32(b[4 * h + j]) * mul;
      if constexpr (INT8) {
        w[h] = pack4_low(round_away(x[0]), round_away(x[1]), round_away(x[2]), round_away(x[3]));
      } else {
        w[h] = pack4_e4m3(clampf(x[0], -448.f, 448.f), clampf(x[1], -448.f, 448.f), clampf(x[2], -448.f, 448.f),
                          clampf(x[3], -448.f, 448.f));
      }
    }
    *((v2i*)dst + i) = v2i{(int)w[0], (int)w[1]};
  }
}

constexpr int64_t ROW_QUANT_MAX_HIDDEN = 1024 * 8 * 4;  // the longest row that 1024 lanes keep in registers

// Launches row_quant_body over `rows` rows of 16-bit values (quant.hip); hidden <= ROW_QUANT_MAX_HIDDEN, % 8 == 0.
int launch_row_quant(const RowQuantArgs& a, int64_t rows, int in_dtype, bool int8, bool silu, hipStream_t st);

}  // namespace sglamd
