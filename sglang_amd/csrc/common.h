// Shared device/host helpers for the gfx950 quantized-linear kernels.
// Everything here is HIP for CDNA4 (wave64); there is no other target.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/sglamd.h"

namespace sglamd {

// Records a message retrievable through sglamd_last_error() and returns `code`.
int fail(int code, const char* fmt, ...);

#define SGLAMD_REQUIRE(cond, code, ...) \
  do {                                  \
    if (!(cond)) return ::sglamd::fail((code), __VA_ARGS__); \
  } while (0)

// Turns the status of the launch that just happened into a C-ABI return code.
int check_launch(const char* what);

typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef unsigned short u16;

__device__ __forceinline__ float bf16_bits_to_f32(u16 h) { return __uint_as_float(((uint32_t)h) << 16); }

// fp32 -> bf16 bits, round-to-nearest-even, NaN kept quiet: gfx950 converts in hardware (v_cvt_pk_bf16_f32),
// one instruction where the bit arithmetic takes seven.
__device__ __forceinline__ u16 f32_to_bf16_bits(float f) {
  const __bf16 b = (__bf16)f;
  u16 h;
  __builtin_memcpy(&h, &b, 2);
  return h;
}
// two at once: low half a, high half b
__device__ __forceinline__ uint32_t f32x2_to_bf16x2_bits(float a, float b) {
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  typedef float f32x2_t __attribute__((ext_vector_type(2)));
  const bf16x2_t p = __builtin_convertvector((f32x2_t){a, b}, bf16x2_t);
  uint32_t w;
  __builtin_memcpy(&w, &p, 4);
  return w;
}

__device__ __forceinline__ float f16_bits_to_f32(u16 h) {
  _Float16 v;
  __builtin_memcpy(&v, &h, 2);
  return (float)v;
}

__device__ __forceinline__ u16 f32_to_f16_bits(float f) {
  _Float16 v = (_Float16)f;  // v_cvt_f16_f32: round-to-nearest-even
  u16 h;
  __builtin_memcpy(&h, &v, 2);
  return h;
}

// 16-bit storage tags used to pick the conversion at compile time.
struct BF16 {
  static constexpr int tag = SGLAMD_BF16;
  typedef u16 storage;
  static __device__ __forceinline__ float to_f32(u16 h) { return bf16_bits_to_f32(h); }
  static __device__ __forceinline__ u16 from_f32(float f) { return f32_to_bf16_bits(f); }
  static __device__ __forceinline__ uint32_t pack2(float a, float b) { return f32x2_to_bf16x2_bits(a, b); }
};
struct F16 {
  static constexpr int tag = SGLAMD_F16;
  typedef u16 storage;
  static __device__ __forceinline__ float to_f32(u16 h) { return f16_bits_to_f32(h); }
  static __device__ __forceinline__ u16 from_f32(float f) { return f32_to_f16_bits(f); }
  static __device__ __forceinline__ uint32_t pack2(float a, float b) {
    return (uint32_t)f32_to_f16_bits(a) | ((uint32_t)f32_to_f16_bits(b) << 16);
  }
};
struct F32 {
  static constexpr int tag = SGLAMD_F32;
  typedef float storage;
  static __device__ __forceinline__ float to_f32(float h) { return h; }
  static __device__ __forceinline__ float from_f32(float f) { return f; }
};

// Two fp32 -> two OCP e4m3fn bytes in the low half of the result (v_cvt_pk_fp8_f32,
// round-to-nearest-even; callers clamp to +-448 first, so the overflow behaviour of the
// instruction never matters).
__device__ __forceinline__ uint32_t pack2_e4m3(float a, float b) {
  return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false) & 0xffffu;
}
__device__ __forceinline__ uint32_t pack4_e4m3(float a, float b, float c, float d) {
  int w = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false);
  w = __builtin_amdgcn_cvt_pk_fp8_f32(c, d, w, true);
  return (uint32_t)w;
}

__device__ __forceinline__ float clampf(float v, float lo, float hi) { return fminf(fmaxf(v, lo), hi); }

// silu(x) = x / (1 + exp(-x)) rounded to the 16-bit type T, as fp32.
//
// The value is defined through expf and the IEEE division, about 30 VALU instructions, and a kernel that reads 16-bit
// gates from HBM is then bound by them and not by the memory.  For bfloat16 the hardware's exp2 (its argument split in
// two, so that its error does not grow with x) and reciprocal, 1 ulp each, give the same 16-bit value unless the fp32
// result lies next to a rounding boundary: the two forms differ by at most 1 + 1/2 (exp2 and its correction) + 1/2 (1 +)
// + 1 (rcp) + 1/2 (*) and 1 + 1/2 + 1/2 (the defined form) times 2^-23, eleven units in the last place, so results within
// D = 16 units of a boundary, one in two thousand, take the defined form.  So do the ranges where that count does not
// hold: below -60 (the reciprocal's subnormals), above 1e30 (the product with log2 e overflows), NaN.
// A half lies next to a boundary eight times as often, and the sign of its zeros is decided by which instruction the
// compiler picks for the product behind it (v_fma_mixlo_f16 adds a +0), so it keeps the defined form.
template <typename T>
__device__ __forceinline__ float silu_rounded(float x) {
  if constexpr (T::tag == SGLAMD_BF16) {
    constexpr uint32_t TIE = 0x8000u, MASK = 0xffffu, D = 16;
    constexpr float L2E_HI = 1.44269502162933349609375f, L2E_LO = 1.9259629911e-8f, LN2 = 0.69314718055994530942f;
    const float p = x * -L2E_HI;
    const float rest = fmaf(x, -L2E_LO, fmaf(x, -L2E_HI, -p));
    const float t = __builtin_amdgcn_exp2f(p);
    float y = x * __builtin_amdgcn_rcpf(1.0f + fmaf(t, rest * LN2, t));
    const bool near_tie = ((__float_as_uint(y) - (TIE - D)) & MASK) <= 2 * D;
    if (near_tie || !(x > -60.f && x < 1e30f)) y = x / (1.0f + expf(-x));
    return T::to_f32(T::from_f32(y));
  } else {
    return T::to_f32(T::from_f32(x / (1.0f + expf(-x))));
  }
}

// Maximum over each aligned group of N = 4, 8 or 16 lanes, in all of them, on the DPP data path.
template <int N>
__device__ __forceinline__ float lanes_max(float v) {
  int x = __float_as_int(v);
#define SGLAMD_DPP_MAX(ctrl) \
  x = __float_as_int(fmaxf(__int_as_float(x), __int_as_float(__builtin_amdgcn_update_dpp(x, x, ctrl, 0xf, 0xf, false))))
  SGLAMD_DPP_MAX(0xB1);               // quad_perm [1, 0, 3, 2]
  SGLAMD_DPP_MAX(0x4E);               // quad_perm [2, 3, 0, 1]
  if (N >= 8) SGLAMD_DPP_MAX(0x141);  // row_half_mirror
  if (N >= 16) SGLAMD_DPP_MAX(0x140);  // row_mirror
#undef SGLAMD_DPP_MAX
  return __int_as_float(x);
}

// Maximum over the wave, in all lanes: within rows of 16 lanes by DPP, the four rows by v_readlane (a shuffle through
// LDS costs a round trip of about 60 cycles for each of its six steps).
__device__ __forceinline__ float wave_max(float v) {
  const int x = __float_as_int(lanes_max<16>(v));
  const float a = __int_as_float(__builtin_amdgcn_readlane(x, 0)), b = __int_as_float(__builtin_amdgcn_readlane(x, 16));
  const float c = __int_as_float(__builtin_amdgcn_readlane(x, 32)), d = __int_as_float(__builtin_amdgcn_readlane(x, 48));
  return fmaxf(fmaxf(a, b), fmaxf(c, d));
}

// One round of a router's top-k over scores v[j] of expert lane + 64 * j: the largest score, the lowest expert among
// those that have it (`fallback` when nothing compares equal: NaN scores); its score is replaced by `taken`.
template <int EPL>
__device__ __forceinline__ float wave_pick(float (&v)[EPL], int fallback, float taken, int& expert) {
  float best = v[0];
#pragma unroll
  for (int j = 1; j < EPL; j++) best = fmaxf(best, v[j]);
  best = wave_max(best);
  int e = -1;
#pragma unroll
  for (int j = 0; j < EPL; j++) {
    const unsigned long long m = __ballot(v[j] == best);
    if (e < 0 && m) e = (int)__builtin_ctzll(m) + 64 * j;
  }
  expert = e < 0 ? fallback : e;
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int j = 0; j < EPL; j++)
    if (lane + 64 * j == expert) v[j] = taken;
  return best;
}

// n / d for 0 <= n < 2^31 and a divisor known on the host: one 32 x 32 -> high 32 bit multiply, an add and a shift
// (T. Granlund and P. Montgomery, Division by Invariant Integers using Multiplication, 1994: the round-up method).
// A 64-bit division by a kernel argument is over a hundred instructions.
struct FastDiv {
  uint32_t mul, shift;
  static FastDiv of(uint32_t d) {
    uint32_t s = 0;
    while (s < 31 && (1u << s) < d) s++;
    return {(uint32_t)((((uint64_t)1 << 32) * (((uint64_t)1 << s) - d)) / d + 1), s};
  }
  __host__ __device__ uint32_t divide(uint32_t n) const {
    return (uint32_t)((((uint64_t)n * mul) >> 32) + n) >> shift;
  }
};

static inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// The current device, asked for once per entry point: while a DeviceScope is alive on a thread its launches share one
// hipGetDevice (the cost models of a single decode GEMM used to make about a hundred of them, 2 us).  Nothing between an
// entry point's first and last launch changes the device.
inline thread_local int scoped_device = -1;
struct DeviceScope {
  const int outer;
  DeviceScope() : outer(scoped_device) {
    if (outer < 0 && hipGetDevice(&scoped_device) != hipSuccess) scoped_device = -1;
  }
  ~DeviceScope() { scoped_device = outer; }
  DeviceScope(const DeviceScope&) = delete;
};
static inline int current_device() {  // -1 when the query fails
  if (scoped_device >= 0) return scoped_device;
  int dev = 0;
  return hipGetDevice(&dev) == hipSuccess ? dev : -1;
}

// Compute units of the current device (cached per device; 256 when the query fails, the MI355X count).
static inline int device_cus() {
  static int cus[32] = {};
  const int dev = current_device();
  if (dev < 0 || dev >= 32) return 256;
  if (!cus[dev]) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cus[dev] = n;
  }
  return cus[dev];
}

// A kernel that asks for more than 64 KB of dynamic LDS needs hipFuncAttributeMaxDynamicSharedMemorySize
// raised once per device; `state` is one object per kernel instantiation (a function-local static).
struct SmemAttrOnce {
  int bytes[32] = {};
};
static inline hipError_t raise_dynamic_smem(SmemAttrOnce& state, const void* kern, int bytes) {
  const int dev = current_device();
  const bool cached = dev >= 0 && dev < 32;
  if (cached && state.bytes[dev] >= bytes) return hipSuccess;
  const hipError_t e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (e == hipSuccess && cached) state.bytes[dev] = bytes;
  return e;
}

}  // namespace sglamd
