// Dense 8-bit GEMM entry points: block-scaled FP8 and INT8, per-token/per-channel FP8 and INT8.  The kernels are
// instantiated in gemm_mode_*.hip (one scaling mode each); this file validates arguments and hands over.
#include "gemm_dispatch.h"

namespace sglamd {

thread_local int last_kernel = 0;
thread_local int skinny_last_shape = 0;
thread_local int strip_last_shape = 0;

extern template int dispatch_out<GEMM_BLOCK_FP8>(const GemmArgs&, int, hipStream_t, void*, int64_t);
extern template int dispatch_out_biased<GEMM_BLOCK_FP8>(const GemmArgs&, int, hipStream_t, void*, int64_t);
extern template int dispatch_quantising<GEMM_BLOCK_FP8, false>(const GemmArgs&, int, hipStream_t, bool);
extern template int dispatch_quantising<GEMM_BLOCK_FP8, true>(const GemmArgs&, int, hipStream_t, bool);
extern template int dispatch_quantising<GEMM_ROW_FP8, false>(const GemmArgs&, int, hipStream_t, bool);
extern template int dispatch_out<GEMM_ROW_FP8>(const GemmArgs&, int, hipStream_t, void*, int64_t);
extern template int dispatch_out<GEMM_ROW_INT8>(const GemmArgs&, int, hipStream_t, void*, int64_t);
extern template int dispatch_out<GEMM_BLOCK_INT8>(const GemmArgs&, int, hipStream_t, void*, int64_t);

static int check_common(const char* op, const void* a, const void* b, const void* c, int64_t M, int64_t N, int64_t K,
                        int64_t lda, int64_t ldb, int64_t ldc) {
  SGLAMD_REQUIRE(a && b && c, SGLAMD_EINVAL, "%s: null pointer", op);
  SGLAMD_REQUIRE(M >= 0 && N > 0 && K > 0, SGLAMD_EINVAL, "%s: bad sizes M=%lld N=%lld K=%lld", op, (long long)M,
                 (long long)N, (long long)K);
  SGLAMD_REQUIRE(M < (1ll << 31) && N < (1ll << 31) && K < (1ll << 31), SGLAMD_EINVAL, "%s: size exceeds int32", op);
  SGLAMD_REQUIRE(K % 16 == 0, SGLAMD_EINVAL, "%s: K (%lld) must be a multiple of 16 bytes", op, (long long)K);
  SGLAMD_REQUIRE(lda >= K && ldb >= K && ldc >= N, SGLAMD_EINVAL, "%s: leading dimension smaller than the row", op);
  SGLAMD_REQUIRE(lda % 16 == 0 && ldb % 16 == 0, SGLAMD_EINVAL, "%s: row strides must be multiples of 16 bytes", op);
  SGLAMD_REQUIRE(((uintptr_t)a % 16) == 0 && ((uintptr_t)b % 16) == 0, SGLAMD_EINVAL,
                 "%s: operands must be 16-byte aligned", op);
  return SGLAMD_OK;
}

}  // namespace sglamd

using namespace sglamd;

static int blockwise(int mode, const char* op, const void* a, int64_t lda, const void* b, int64_t ldb, const float* sa,
                     int64_t sa_stride_m, int64_t sa_stride_k, const float* sb, int64_t sb_stride_n,
                     int64_t sb_stride_k, void* out, int64_t ldc, int out_dtype, int64_t M, int64_t N, int64_t K,
                     void* workspace, int64_t workspace_bytes, void* stream, bool scales_pow2 = false,
                     const void* bias = nullptr) {
  const DeviceScope scope;
  int rc = check_common(op, a, b, out, M, N, K, lda, ldb, ldc);
  if (rc) return rc;
  SGLAMD_REQUIRE(sa && sb, SGLAMD_EINVAL, "%s: null scale pointer", op);
  if (M == 0) return SGLAMD_OK;
  GemmArgs g = {};
  g.scales_pow2 = scales_pow2;
  g.A = (const uint8_t*)a;
  g.lda = lda;
  g.B = (const uint8_t*)b;
  g.ldb = ldb;
  g.sa = sa;
  g.sa_sm = sa_stride_m;
  g.sa_sk = sa_stride_k;
  g.sb = sb;
  g.sb_sn = sb_stride_n;
  g.sb_sk = sb_stride_k;
  g.C = out;
  g.ldc = ldc;
  g.M = (int)M;
  g.N = (int)N;
  g.K = (int)K;
  g.bias = bias;
  if (mode == GEMM_BLOCK_FP8 && bias)
    return dispatch_out_biased<GEMM_BLOCK_FP8>(g, out_dtype, (hipStream_t)stream, workspace, workspace_bytes);
  if (mode == GEMM_BLOCK_FP8)
    return dispatch_out<GEMM_BLOCK_FP8>(g, out_dtype, (hipStream_t)stream, workspace, workspace_bytes);
  return dispatch_out<GEMM_BLOCK_INT8>(g, out_dtype, (hipStream_t)stream, workspace, workspace_bytes);
}

extern "C" int sglamd_fp8_blockwise_scaled_mm(const void* a, int64_t lda, const void* b, int64_t ldb, const float* sa,
                                              int64_t sa_stride_m, int64_t sa_stride_k, const float* sb,
                                              int64_t sb_stride_n, int64_t sb_stride_k, void* out, int64_t ldc,
                                              int out_dtype, int64_t M, int64_t N, int64_t K, void* workspace,
                                              int64_t workspace_bytes, void* stream) {
  return blockwise(GEMM_BLOCK_FP8, "fp8_blockwise_scaled_mm", a, lda, b, ldb, sa, sa_stride_m, sa_stride_k, sb,
                   sb_stride_n, sb_stride_k, out, ldc, out_dtype, M, N, K, workspace, workspace_bytes, stream);
}

extern "C" int sglamd_fp8_blockwise_scaled_mm_pow2(const void* a, int64_t lda, const void* b, int64_t ldb,
                                                   const float* sa, int64_t sa_stride_m, int64_t sa_stride_k,
                                                   const float* sb, int64_t sb_stride_n, int64_t sb_stride_k, void* out,
                                                   int64_t ldc, int out_dtype, int64_t M, int64_t N, int64_t K,
                                                   void* workspace, int64_t workspace_bytes, void* stream) {
  return blockwise(GEMM_BLOCK_FP8, "fp8_blockwise_scaled_mm_pow2", a, lda, b, ldb, sa, sa_stride_m, sa_stride_k, sb,
                   sb_stride_n, sb_stride_k, out, ldc, out_dtype, M, N, K, workspace, workspace_bytes, stream, true);
}

extern "C" int sglamd_fp8_blockwise_scaled_mm_bias(const void* a, int64_t lda, const void* b, int64_t ldb,
                                                   const float* sa, int64_t sa_stride_m, int64_t sa_stride_k,
                                                   const float* sb, int64_t sb_stride_n, int64_t sb_stride_k,
                                                   int scales_pow2, const void* bias, void* out, int64_t ldc,
                                                   int out_dtype, int64_t M, int64_t N, int64_t K, void* workspace,
                                                   int64_t workspace_bytes, void* stream) {
  SGLAMD_REQUIRE(bias && ((uintptr_t)bias & 1) == 0, SGLAMD_EINVAL, "fp8_blockwise_scaled_mm_bias: null or odd bias pointer");
  return blockwise(GEMM_BLOCK_FP8, "fp8_blockwise_scaled_mm_bias", a, lda, b, ldb, sa, sa_stride_m, sa_stride_k, sb,
                   sb_stride_n, sb_stride_k, out, ldc, out_dtype, M, N, K, workspace, workspace_bytes, stream,
                   scales_pow2 != 0, bias);
}

// Linear layers of up to this many rows may quantise them in the GEMM's own workgroups (0: none).  The kernel holds one tile of 16.
static int quantising_max_rows() {
  static const int v = getenv("SGLAMD_LINEAR_FUSE_ROWS") ? atoi(getenv("SGLAMD_LINEAR_FUSE_ROWS")) : 16;  // tuning knob
  return v < 16 ? v : 16;
}
// Which of them do.  A launch less saves 1-2 us; every workgroup quantising every row costs it time that grows with M * K
// and delays its weight stream.  Two launches -> one, us, weights from HBM, queue kept full, block scales (row scales):
//   one row    36864 x 7168 42.6 -> 41.2, 7168 x 16384 21.9 -> 21.4, 24576 x 1536 10.9 -> 8.9 (11.2 -> 9.5), 4096 x 4096 7.5 -> 6.3
//              (8.1 -> 6.7), 1024 x 7168 8.3 -> 6.6 (8.7 -> 6.9), (10240 x 8192 17.8 -> 16.7)
//   two rows   36864 x 7168 42.6 -> 42.1, 24576 x 1536 10.6 -> 8.6 (11.0 -> 9.1), 4096 x 4096 7.6 -> 6.4 (7.9 -> 6.9), 1024 x 7168 8.3 -> 7.2
//   three      36864 x 7168 42.7 -> 42.9, 1024 x 7168 8.4 -> 7.9 (8.8 -> 8.6), (10240 x 8192 17.9 -> 18.9)
//   four       36864 x 7168 42.7 -> 43.4, 24576 x 1536 10.8 -> 9.0 (11.0 -> 9.8), 4096 x 4096 7.6 -> 7.0 (7.9 -> 7.7), 1024 x 1024 7.2 -> 5.5
//   eight      24576 x 1536 10.8 -> 9.6 (11.3 -> 10.7), 4096 x 4096 7.8 -> 8.4, 1024 x 1024 7.1 -> 6.0 (7.6 -> 6.8), 4096 x 2048 7.6 -> 7.2
//              (7.5 -> 7.7)
//   sixteen    4096 x 512 6.9 -> 6.0 (7.8 -> 7.3), 1024 x 1024 7.3 -> 6.9 (7.6 -> 8.1)
// and of a call that the host launches in 9.5 us (10) with an empty queue, 2.5 us: 1024 x 1024 at four to twelve rows 9.5 -> 6.5 (10 -> 7).
static bool linear_quantises(int64_t M, int64_t K, bool row_scales) {
  return M >= 1 && M <= quantising_max_rows() && (M == 1 || M * K <= (M > 4 && row_scales ? 12288 : 16384));
}

extern "C" int sglamd_fp8_block_linear(const void* x, int dtype, int64_t M, int64_t K, const void* w, int64_t ldb,
                                       const float* sb, int64_t sb_stride_n, int64_t sb_stride_k, const void* bias,
                                       void* out, int64_t ldc, int64_t N, void* q, float* sa, void* workspace,
                                       int64_t workspace_bytes, void* stream) {
  const char* op = "fp8_block_linear";
  SGLAMD_REQUIRE(x && w && sb && out && q && sa, SGLAMD_EINVAL, "%s: null pointer", op);
  SGLAMD_REQUIRE(dtype == SGLAMD_BF16 || dtype == SGLAMD_F16, SGLAMD_EINVAL, "%s: dtype must be Half or BFloat16", op);
  SGLAMD_REQUIRE(K > 0 && K % 128 == 0, SGLAMD_EINVAL, "%s: K (%lld) must be a positive multiple of 128", op, (long long)K);
  SGLAMD_REQUIRE(!bias || ((uintptr_t)bias & 1) == 0, SGLAMD_EINVAL, "%s: odd bias pointer", op);
  const DeviceScope scope;
  if (linear_quantises(M, K, false) && ((uintptr_t)x % 16) == 0) {
    int rc = check_common(op, x, w, out, M, N, K, K, ldb, ldc);
    if (rc) return rc;
    GemmArgs g = {};
    g.A16 = x;
    g.lda16 = K * 2;
    g.act_mode = 1;
    g.q_eps = 1e-10f;
    g.q_min = -448.f;
    g.q_max = 448.f;
    g.lda = K;
    g.B = (const uint8_t*)w;
    g.ldb = ldb;
    g.sb = sb;
    g.sb_sn = sb_stride_n;
    g.sb_sk = sb_stride_k;
    g.C = out;
    g.ldc = ldc;
    g.M = (int)M;
    g.N = (int)N;
    g.K = (int)K;
    g.bias = bias;
    if (gemm8_skinny_ok(g, M) && (bias ? dispatch_quantising<GEMM_BLOCK_FP8, true> : dispatch_quantising<GEMM_BLOCK_FP8, false>)(g, dtype, (hipStream_t)stream, false))
      return (bias ? dispatch_quantising<GEMM_BLOCK_FP8, true> : dispatch_quantising<GEMM_BLOCK_FP8, false>)(g, dtype, (hipStream_t)stream, true);
  }
  const int rc = sglamd_per_token_group_quant_8bit(x, dtype, q, SGLAMD_FP8_E4M3, sa, M, K, 128, SGLAMD_SCALE_COL_MAJOR, M, 1e-10f,
                                                   -448.f, 448.f, SGLAMD_QUANT_FORM_RECIPROCAL, stream);
  if (rc) return rc;
  return blockwise(GEMM_BLOCK_FP8, op, q, K, w, ldb, sa, 1, M, sb, sb_stride_n, sb_stride_k, out, ldc, dtype, M, N, K, workspace,
                   workspace_bytes, stream, false, bias);
}

extern "C" int sglamd_int8_blockwise_scaled_mm(const void* a, int64_t lda, const void* b, int64_t ldb, const float* sa,
                                               int64_t sa_stride_m, int64_t sa_stride_k, const float* sb,
                                               int64_t sb_stride_n, int64_t sb_stride_k, void* out, int64_t ldc,
                                               int out_dtype, int64_t M, int64_t N, int64_t K, void* workspace,
                                               int64_t workspace_bytes, void* stream) {
  return blockwise(GEMM_BLOCK_INT8, "int8_blockwise_scaled_mm", a, lda, b, ldb, sa, sa_stride_m, sa_stride_k, sb,
                   sb_stride_n, sb_stride_k, out, ldc, out_dtype, M, N, K, workspace, workspace_bytes, stream);
}

static int rowwise(int mode, const char* op, const void* a, int64_t lda, const void* b, int64_t ldb, const float* sa,
                   const float* sb, const void* bias, void* out, int64_t ldc, int out_dtype, int64_t M, int64_t N,
                   int64_t K, void* workspace, int64_t workspace_bytes, void* stream) {
  const DeviceScope scope;
  int rc = check_common(op, a, b, out, M, N, K, lda, ldb, ldc);
  if (rc) return rc;
  SGLAMD_REQUIRE(sa && sb, SGLAMD_EINVAL, "%s: null scale pointer", op);
  if (M == 0) return SGLAMD_OK;
  GemmArgs g = {};
  g.A = (const uint8_t*)a;
  g.lda = lda;
  g.B = (const uint8_t*)b;
  g.ldb = ldb;
  g.sa = sa;
  g.sb = sb;
  g.bias = bias;
  g.C = out;
  g.ldc = ldc;
  g.M = (int)M;
  g.N = (int)N;
  g.K = (int)K;
  if (mode == GEMM_ROW_FP8) return dispatch_out<GEMM_ROW_FP8>(g, out_dtype, (hipStream_t)stream, workspace, workspace_bytes);
  return dispatch_out<GEMM_ROW_INT8>(g, out_dtype, (hipStream_t)stream, workspace, workspace_bytes);
}

extern "C" int sglamd_fp8_scaled_mm(const void* a, int64_t lda, const void* b, int64_t ldb, const float* sa,
                                    const float* sb, const void* bias, void* out, int64_t ldc, int out_dtype,
                                    int64_t M, int64_t N, int64_t K, void* workspace, int64_t workspace_bytes,
                                    void* stream) {
  return rowwise(GEMM_ROW_FP8, "fp8_scaled_mm", a, lda, b, ldb, sa, sb, bias, out, ldc, out_dtype, M, N, K, workspace,
                 workspace_bytes, stream);
}

extern "C" int sglamd_fp8_row_linear(const void* x, int dtype, int64_t M, int64_t K, const void* w, int64_t ldb, const float* sb,
                                     const void* bias, void* out, int64_t ldc, int64_t N, void* q, float* sa, void* workspace,
                                     int64_t workspace_bytes, void* stream) {
  const char* op = "fp8_row_linear";
  SGLAMD_REQUIRE(x && w && sb && out && q && sa, SGLAMD_EINVAL, "%s: null pointer", op);
  SGLAMD_REQUIRE(dtype == SGLAMD_BF16 || dtype == SGLAMD_F16, SGLAMD_EINVAL, "%s: dtype must be Half or BFloat16", op);
  const DeviceScope scope;
  if (linear_quantises(M, K, true) && K % 128 == 0 && ((uintptr_t)x % 16) == 0) {
    int rc = check_common(op, x, w, out, M, N, K, K, ldb, ldc);
    if (rc) return rc;
    GemmArgs g = {};
    g.A16 = x;
    g.lda16 = K * 2;
    g.act_mode = 1;
    g.q_min = -448.f;
    g.q_max = 448.f;
    g.lda = K;
    g.B = (const uint8_t*)w;
    g.ldb = ldb;
    g.sb = sb;
    g.bias = bias;
    g.C = out;
    g.ldc = ldc;
    g.M = (int)M;
    g.N = (int)N;
    g.K = (int)K;
    if (gemm8_skinny_ok(g, M) && dispatch_quantising<GEMM_ROW_FP8, false>(g, dtype, (hipStream_t)stream, false))
      return dispatch_quantising<GEMM_ROW_FP8, false>(g, dtype, (hipStream_t)stream, true);
  }
  const int rc = sglamd_per_token_quant_fp8(x, dtype, q, sa, M, K, stream);
  if (rc) return rc;
  return rowwise(GEMM_ROW_FP8, op, q, K, w, ldb, sa, sb, bias, out, ldc, dtype, M, N, K, workspace, workspace_bytes, stream);
}

extern "C" int sglamd_int8_scaled_mm(const void* a, int64_t lda, const void* b, int64_t ldb, const float* sa,
                                     const float* sb, const void* bias, void* out, int64_t ldc, int out_dtype,
                                     int64_t M, int64_t N, int64_t K, void* workspace, int64_t workspace_bytes,
                                     void* stream) {
  return rowwise(GEMM_ROW_INT8, "int8_scaled_mm", a, lda, b, ldb, sa, sb, bias, out, ldc, out_dtype, M, N, K, workspace,
                 workspace_bytes, stream);
}

extern "C" int sglamd_last_gemm_kernel(void) { return last_kernel; }
extern "C" int sglamd_last_streaming_shape(void) { return skinny_last_shape; }
extern "C" int sglamd_last_strip_shape(void) { return strip_last_shape; }

extern "C" int sglamd_dense_plan(int block_scales, int64_t M, int64_t N, int64_t K, int32_t* plan) {
  const char* op = "dense_plan";
  SGLAMD_REQUIRE(plan, SGLAMD_EINVAL, "%s: null pointer", op);
  SGLAMD_REQUIRE(M > 0 && N > 0 && K > 0 && M < (1ll << 31) && N < (1ll << 31) && K < (1ll << 31), SGLAMD_EINVAL, "%s: sizes out of range", op);
  const DeviceScope scope;
  return dense_plan(block_scales != 0, M, N, K, plan);
}

extern "C" int sglamd_streaming_piece_offset(int kb, int lchunk, int64_t K, int64_t* offset) {
  const SkinnyPiece pc = skinny_piece(kb, lchunk, (int)K);
  if (offset) *offset = pc.offset;
  return pc.dead ? 1 : 0;
}

// Bytes of fp32 scratch with which the GEMM entry points above can split K for this shape (0: no use for it).
extern "C" int64_t sglamd_gemm_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  if (M >= (1ll << 31) || N <= 0 || K <= 0) return 0;
  const DeviceScope scope;
  const DenseChoice choice = dense_choice(M, N, K);
  if (choice.row_tile) return 0;
  if (choice.strip.rows) return choice.strip.slices > 1 ? (int64_t)choice.strip.slices * M * N * 4 : 0;
  if (M <= 64 && !small_m_uses_tile(M, N, K)) return 0;
  const BigConfig cfg = gemm8_big_config(M, N, K);
  int64_t need = cfg.slices > 1 ? (int64_t)cfg.slices * M * N * 4 : 0;
  // a launch of 256-row tiles cut in two along N (column_split) splits K on its second part; whether the launch
  // uses 256-row tiles depends on the operand mode, so the larger of the two needs is reported
  const int64_t n1 = M > 64 ? column_split(M, N, K) : 0;
  if (n1 > 0) {
    const int64_t rest = (int64_t)gemm8_big_config(M, N - n1, K).slices * M * (N - n1) * 4;
    if (rest > need) need = rest;
  }
  return need;
}
