// The host side of the path as native code: the torch.ops.sgl_kernel operators and the whole-call functions behind
// the Python wrappers (sglang_amd._C).  Everything on the GPU is in libsglamd.so; this file checks tensors, allocates
// outputs and scratch from torch's caching allocator and calls the C ABI on torch's current stream.
//
// Why it is native: a decode-sized linear layer is 15-25 us of kernels, and the same checks, allocations and ctypes
// calls made from Python took 15-18 us for each of its launches, so that the host set the pace (an o_proj of one
// token: 36 us a call for 22.7 us of kernels).
//
// Two kinds of functions:
//   * operators, with the schema strings and the error texts of sgl-kernel (csrc/common_extension.cc:76-77,116-142,
//     164-181), registered for device tensors;
//   * calls that stand for a whole Python wrapper (quantise + GEMM, a MoE layer).  They take the plain configurations
//     and answer "not mine" (an empty optional, None in Python) for anything else, before any work: the wrapper then
//     goes through its steps one by one, which also raise the errors for arguments that are wrong.
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <torch/extension.h>

#include "../../include/sglamd.h"

namespace {

using at::ScalarType;
using at::Tensor;
using c10::optional;

PyObject* g_error_type = nullptr;  // sglang_amd._lib.SglAmdError

void check(int rc) {
  if (rc == SGLAMD_OK) return;
  const std::string msg = sglamd_last_error();
  if (rc == SGLAMD_ENOTSUP) C10_THROW_ERROR(NotImplementedError, msg);
  py::gil_scoped_acquire gil;
  PyErr_SetString(g_error_type ? g_error_type : PyExc_RuntimeError, msg.c_str());
  throw py::error_already_set();
}

void* stream_of(const Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

bool is_half(ScalarType t) { return t == at::kHalf || t == at::kBFloat16; }

int tag(ScalarType t) {
  switch (t) {
    case at::kFloat: return SGLAMD_F32;
    case at::kHalf: return SGLAMD_F16;
    case at::kBFloat16: return SGLAMD_BF16;
    case ScalarType::Float8_e4m3fn: return SGLAMD_FP8_E4M3;
    case at::kChar: return SGLAMD_I8;
    case at::kInt: return SGLAMD_I32;
    case at::kLong: return SGLAMD_I64;
    default: TORCH_CHECK(false, "unsupported dtype ", t);
  }
}

constexpr ScalarType kFp8 = ScalarType::Float8_e4m3fn;

void check_input(const Tensor& t, const char* name) {
  TORCH_CHECK(t.is_cuda(), name, " must be a CUDA tensor");
  TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
}

// A size that a division below is by: an integer division by zero ends the process with SIGFPE.
void check_positive(int64_t v, const char* name) { TORCH_CHECK(v > 0, name, " must be positive, but got ", v); }

int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }
int64_t up(int64_t a, int64_t b) { return cdiv(a, b) * b; }

// Whether somebody between the dispatcher and the kernels has to see the operators that a whole-call function stands for: a
// dispatch mode (fake tensors, a tracer, functorch) is active on this thread, a tensor is not a plain dense one (a
// subclass with its own dispatch, a transform's wrapper, a lazy conjugate or negation), or autograd records it, backward
// or forward (the addition of a bias carries its gradient; the operators say that they have none).  Then the call is not
// ours.  Below autograd, where a custom operator's implementation runs, nothing is recorded.
bool is_observed() {
  const uint64_t usual = c10::default_included_set.raw_repr();
  return (c10::impl::tls_local_dispatch_key_set().included_.raw_repr() & ~usual) != 0;
}
bool is_observed(const Tensor& t) {
  static const uint64_t plain =
      c10::DispatchKeySet({c10::DispatchKey::CUDA, c10::DispatchKey::AutogradCUDA, c10::DispatchKey::ADInplaceOrView,
                           c10::DispatchKey::AutocastCUDA})
          .raw_repr();
  if ((t.key_set().raw_repr() & ~plain) != 0) return true;
  if (c10::impl::tls_local_dispatch_key_set().excluded_.has_any(c10::autograd_dispatch_keyset)) return false;
  return (c10::GradMode::is_enabled() && t.requires_grad()) || t._fw_grad(/*level=*/0).defined();
}
bool is_observed(const optional<Tensor>& t) { return t && is_observed(*t); }
template <typename... Tensors>
bool any_observed(const Tensors&... tensors) {
  return is_observed() || (is_observed(tensors) || ...);
}

// What an operator that declares the write does for autograd: a tensor saved before it no longer counts as unchanged.
// (Inference tensors have no version.)
void written_in_place(const Tensor& t) {
  if (!t.is_inference()) t.unsafeGetTensorImpl()->bump_version();
}

Tensor empty(at::IntArrayRef shape, ScalarType t, const Tensor& like) {
  return at::empty(shape, at::TensorOptions().dtype(t).device(like.device()));
}

// Scratch of one call: a single allocation whose pieces start at multiples of 256 bytes.
struct Scratch {
  Tensor buf;
  int64_t bytes = 0;
  int64_t take(int64_t n) {
    const int64_t at = bytes;
    bytes += up(n, 256);
    return at;
  }
  void allocate(const Tensor& like) {
    if (bytes) buf = empty({bytes}, at::kByte, like);
  }
  void* at(int64_t offset) const { return (uint8_t*)buf.data_ptr() + offset; }
};

// Stride between the rows of a matrix whose other dimension is contiguous (a 1-row matrix may report any there).
int64_t ld(const Tensor& t, int64_t dim) {
  return t.size(dim) > 1 ? t.stride(dim) : std::max(t.stride(dim), t.size(1 - dim));
}

// ---------------------------------------------------------------------------------------
// activation quantisation
// ---------------------------------------------------------------------------------------
void group_quant(const Tensor& input, const Tensor& q, const Tensor& s, int64_t group, double eps, double lo, double hi,
                 bool ue8m0, int form, bool col_major, bool silu) {
  int64_t hidden = input.size(-1);
  check_positive(hidden, "hidden size");
  const int64_t rows = input.numel() / hidden;
  if (silu) {  // input rows are [gate | up], the quantised row has half the width (v2.cu:412-424)
    TORCH_CHECK(hidden % 2 == 0 && q.size(-1) == hidden / 2, "output_q must have half of input's last dim");
    hidden /= 2;
    TORCH_CHECK(hidden % group == 0, "hidden size must be a multiple of group_size");
  }
  int layout = SGLAMD_SCALE_ROW_MAJOR;
  int64_t stride = 0;
  if (col_major) {
    layout = ue8m0 ? SGLAMD_SCALE_COL_MAJOR_UE8M0 : SGLAMD_SCALE_COL_MAJOR;
    stride = s.stride(-1);
  } else {
    TORCH_CHECK(!ue8m0, "scale_ue8m0 requires column-major scales");
    TORCH_CHECK(s.is_contiguous(), "row-major output_s must be contiguous");
  }
  const ScalarType t = input.scalar_type();
  TORCH_CHECK(t == at::kFloat || is_half(t), "input must be Float, Half or BFloat16");
  TORCH_CHECK(q.scalar_type() == kFp8 || q.scalar_type() == at::kChar, "output_q must be Float8_e4m3fn or Char");
  if (ue8m0) {
    TORCH_CHECK(s.scalar_type() == at::kInt, "UE8M0 output_s must be Int (four exponents per element)");
  } else {
    TORCH_CHECK(s.scalar_type() == at::kFloat, "output_s must be Float32");
  }
  const c10::DeviceGuard guard(input.device());
  auto fn = silu ? sglamd_silu_mul_group_quant_8bit : sglamd_per_token_group_quant_8bit;
  check(fn(input.data_ptr(), tag(t), q.data_ptr(), tag(q.scalar_type()), s.data_ptr(), rows, hidden, (int)group, layout,
           stride, (float)eps, (float)lo, (float)hi, form, stream_of(input)));
}

// per_token_group_quant_8bit.cu:116-217: contiguous inputs, numel % group == 0, 2-D scales, column-major when
// output_s.stride(0) < output_s.stride(1)
void sgl_per_token_group_quant_8bit(const Tensor& input, const Tensor& q, const Tensor& s, int64_t group, double eps,
                                    double lo, double hi, bool ue8m0) {
  check_input(input, "input");
  check_input(q, "output_q");
  check_positive(group, "group_size");
  TORCH_CHECK(input.numel() % group == 0, "input.numel() % group_size must be 0");
  TORCH_CHECK(s.dim() == 2, "output_s.dim() must be 2");
  TORCH_CHECK(input.size(-1) % group == 0, "hidden size must be a multiple of group_size");
  group_quant(input, q, s, group, eps, lo, hi, ue8m0, SGLAMD_QUANT_FORM_DIVIDE, s.stride(0) < s.stride(1), false);
}

// per_token_group_quant_8bit_v2.cu:411-542 (checks :425-447,482-527)
void sgl_per_token_group_quant_8bit_v2(const Tensor& input, const Tensor& q, const Tensor& s, int64_t group, double eps,
                                       double lo, double hi, bool ue8m0, bool silu, const optional<Tensor>& masked_m) {
  check_input(input, "input");
  check_input(q, "output_q");
  TORCH_CHECK(input.numel() > 0, "input.numel() must be > 0");
  TORCH_CHECK(std::abs(1e-10 - eps) < 1e-13, "eps must be 1e-10");
  check_positive(group, "group_size");
  TORCH_CHECK(input.numel() % group == 0, "input.numel() % group_size must be 0");
  const bool masked = masked_m.has_value();
  TORCH_CHECK(s.dim() == (masked ? 3 : 2), "output_s.dim() must be ", masked ? 3 : 2);
  TORCH_CHECK(group == 16 || group == 32 || group == 64 || group == 128, "Unsupported group_size");
  TORCH_CHECK(is_half(input.scalar_type()), "input must be Half or BFloat16");
  if (q.scalar_type() == at::kChar) {
    TORCH_CHECK(lo == -128 && hi == 127, "min_8bit/max_8bit must be -128/127 for int8");
  } else {
    TORCH_CHECK(q.scalar_type() == kFp8, "output_q must be Float8_e4m3fn or Char");
    TORCH_CHECK(lo == -448 && hi == 448, "min_8bit/max_8bit must be -448/448 for float8_e4m3fn");
  }
  if (masked && ue8m0 && silu && s.stride(-2) < s.stride(-1)) {
    // the one combination that walks the masked layout (v2.cu:489-494): [experts, tokens, 2*hidden] input, only the
    // first masked_m[e] tokens of each expert are processed
    TORCH_CHECK(input.dim() == 3 && q.dim() == 3, "masked layout takes [experts, tokens, hidden] tensors");
    const Tensor& mm = *masked_m;
    TORCH_CHECK(mm.scalar_type() == at::kInt && mm.is_cuda() && mm.is_contiguous(),
                "masked_m must be a contiguous CUDA Int tensor");
    const int64_t experts = input.size(0), tokens = input.size(1), hidden2 = input.size(2);
    TORCH_CHECK(mm.numel() == experts, "masked_m must hold one count per local expert");
    TORCH_CHECK(hidden2 % 2 == 0 && q.size(-1) == hidden2 / 2 && q.size(-2) == tokens,
                "output_q must have half of input's last dim");
    TORCH_CHECK((hidden2 / 2) % group == 0, "hidden size must be a multiple of group_size");
    TORCH_CHECK(s.scalar_type() == at::kInt && s.stride(-2) == 1,
                "UE8M0 output_s must be Int (four exponents per element), token-contiguous");
    const c10::DeviceGuard guard(input.device());
    check(sglamd_silu_mul_group_quant_8bit_masked(input.data_ptr(), tag(input.scalar_type()), q.data_ptr(),
                                                  tag(q.scalar_type()), s.data_ptr(), experts, tokens, hidden2 / 2,
                                                  (int)group, s.stride(0), s.stride(-1), mm.data_ptr<int32_t>(),
                                                  (float)eps, (float)lo, (float)hi, stream_of(input)));
    return;
  }
  // every other combination ignores masked_m and walks all tokens (NaiveScheduler, v2.cu:495-510)
  group_quant(input, q, s, group, eps, lo, hi, ue8m0, SGLAMD_QUANT_FORM_RECIPROCAL, s.stride(-2) < s.stride(-1), silu);
}

// per_token_quant_fp8.cu:242-314
void sgl_per_token_quant_fp8(const Tensor& input, const Tensor& q, const Tensor& s) {
  check_input(input, "input");
  check_input(q, "output_q");
  check_input(s, "output_s");
  TORCH_CHECK(input.dim() == 2, "input must be 2D");
  const int64_t rows = input.size(0), hidden = input.size(1);
  TORCH_CHECK(hidden % 4 == 0, "Hidden dimension must be divisible by 4, but got ", hidden);
  TORCH_CHECK(q.scalar_type() == kFp8 && s.scalar_type() == at::kFloat,
              "output_q must be Float8_e4m3fn and output_s Float32");
  TORCH_CHECK(s.numel() == rows, "output_s must hold one scale per token");
  if (rows == 0) return;
  const c10::DeviceGuard guard(input.device());
  check(sglamd_per_token_quant_fp8(input.data_ptr(), tag(input.scalar_type()), q.data_ptr(), s.data_ptr<float>(), rows,
                                   hidden, stream_of(input)));
}

// Launcher of the static per-tensor quantiser (the Triton _static_quant_fp8, fp8_kernel.py:681-721): input
// [rows, hidden] contiguous, scale one float32 on the device, scale_rows an optional float32 [rows] that receives the
// scale once per row.
void static_quant_fp8_(const Tensor& input, const Tensor& q, const Tensor& scale, const optional<Tensor>& scale_rows) {
  check_input(input, "input");
  check_input(q, "output_q");
  TORCH_CHECK(input.dim() == 2 && q.sizes() == input.sizes(), "input and output_q must be 2D of the same shape");
  TORCH_CHECK(q.scalar_type() == kFp8, "output_q must be Float8_e4m3fn");
  TORCH_CHECK(scale.is_cuda() && scale.scalar_type() == at::kFloat && scale.numel() == 1,
              "scale must be one Float32 on the device");
  const int64_t rows = input.size(0), hidden = input.size(1);
  if (scale_rows) {
    TORCH_CHECK(scale_rows->is_cuda() && scale_rows->scalar_type() == at::kFloat && scale_rows->is_contiguous() &&
                    scale_rows->numel() == rows,
                "scale_rows must be a contiguous Float32 tensor of one scale per row");
  }
  TORCH_CHECK(hidden % 8 == 0, "the row length must be a multiple of 8, but got ", hidden);
  if (rows == 0) return;
  const c10::DeviceGuard guard(input.device());
  check(sglamd_static_quant_fp8(input.data_ptr(), tag(input.scalar_type()), q.data_ptr(), scale.data_ptr<float>(),
                                scale_rows ? scale_rows->data_ptr<float>() : nullptr, rows, hidden, stream_of(input)));
}

// scale[0] = max(max|input|, eps) / fp8_max: the scale of dynamic per-tensor quantisation
// (fp8_kernel.py:1675-1685,1719-1726)
void tensor_absmax_scale_(const Tensor& input, const Tensor& scale, double eps, double fp8_max) {
  const ScalarType t = input.scalar_type();
  TORCH_CHECK(input.is_cuda() && input.is_contiguous() && (t == at::kFloat || is_half(t)),
              "input must be a contiguous float32, float16 or bfloat16 CUDA tensor");
  TORCH_CHECK(scale.is_cuda() && scale.scalar_type() == at::kFloat && scale.numel() >= 1,
              "scale must be a Float32 CUDA tensor");
  if (input.numel() == 0) {
    scale.fill_(eps / fp8_max);
    return;
  }
  const c10::DeviceGuard guard(input.device());
  const Tensor ws = empty({1024}, at::kFloat, input);
  check(sglamd_tensor_absmax_scale(input.data_ptr(), tag(t), input.numel(), (float)eps, (float)fp8_max,
                                   scale.data_ptr<float>(), ws.data_ptr<float>(), stream_of(input)));
}

// In-place launcher of the per-token INT8 quantiser (int8_kernel.py:28-89 is a Triton kernel in the reference, so
// there is no sgl_kernel schema to mirror)
void per_token_quant_int8_(const Tensor& input, const Tensor& q, const Tensor& s) {
  check_input(input, "input");
  check_input(q, "output_q");
  check_input(s, "output_s");
  const int64_t hidden = input.size(-1), rows = hidden ? input.numel() / hidden : 0;
  if (rows == 0) return;
  const c10::DeviceGuard guard(input.device());
  check(sglamd_per_token_quant_int8(input.data_ptr(), tag(input.scalar_type()), (int8_t*)q.data_ptr(),
                                    (float*)s.data_ptr(), rows, hidden, stream_of(input)));
}

// fp32 [rows, groups] scales out of int32 words of four UE8M0 exponent bytes each: row r reads row r * row_step of
// `packed` ([packed_rows, ceil(groups/4)], any strides); fp8_utils.py:1348-1383
Tensor ue8m0_unpack_(const Tensor& packed, int64_t rows, int64_t groups, int64_t row_step) {
  TORCH_CHECK(packed.is_cuda() && packed.scalar_type() == at::kInt && packed.dim() == 2,
              "packed scales must be a 2D CUDA Int tensor");
  TORCH_CHECK(packed.size(1) * 4 >= groups && (rows == 0 || packed.size(0) > (rows - 1) * row_step),
              "packed scales do not cover the requested rows and groups");
  const c10::DeviceGuard guard(packed.device());
  Tensor out = empty({rows, groups}, at::kFloat, packed);
  check(sglamd_ue8m0_unpack(packed.data_ptr(), packed.stride(0), packed.stride(1), row_step, out.data_ptr<float>(), rows,
                            groups, stream_of(packed)));
  return out;
}

// Scale buffer in one of the four layouts of fp8_kernel.py:454-495 (row-major; column-major with the rows unpadded or
// padded to 4; packed UE8M0 words, groups always 128 wide) for rows of `cols` values.
Tensor scale_buffer(const Tensor& like, int64_t rows, int64_t cols, int64_t group, bool col_major, bool aligned,
                    bool ue8m0) {
  if (ue8m0) {
    const int64_t words = up(cols / 128, 4) / 4, pad = up(rows, 4);
    const Tensor storage = empty({words, pad}, at::kInt, like);
    return storage.as_strided({rows, words}, {1, pad});
  }
  const int64_t groups = cols / group;
  if (!col_major) return empty({rows, groups}, at::kFloat, like);
  const int64_t pad = aligned ? up(rows, 4) : rows;
  const Tensor storage = empty({groups, pad}, at::kFloat, like);
  return storage.as_strided({rows, groups}, {1, pad});
}

// sglang_per_token_group_quant_fp8 / _int8 for a 2-D half-precision input in the reciprocal arithmetic.
optional<std::tuple<Tensor, Tensor>> group_quant_2d(const Tensor& x, int64_t group, double eps, bool col_major,
                                                    bool aligned, bool ue8m0, bool silu, bool int8) {
  if (any_observed(x)) return {};
  if (x.dim() != 2 || !x.is_cuda() || !is_half(x.scalar_type()) || !x.is_contiguous()) return {};
  if (group != 16 && group != 32 && group != 64 && group != 128) return {};
  const int64_t rows = x.size(0), width = silu ? x.size(1) / 2 : x.size(1);
  if (rows == 0 || width == 0 || (silu && x.size(1) % 2) || width % group || std::abs(1e-10 - eps) >= 1e-13) return {};
  if (ue8m0 && !(col_major && aligned && width >= 128)) return {};
  const c10::DeviceGuard guard(x.device());
  Tensor q = empty({rows, width}, int8 ? at::kChar : kFp8, x);
  Tensor s = scale_buffer(x, rows, width, group, col_major, aligned, ue8m0);
  // a buffer whose two strides do not order it (one row or one group) counts as row-major, as in the operator
  const bool col = s.stride(-2) < s.stride(-1);
  if (!col && (ue8m0 || !s.is_contiguous())) return {};
  group_quant(x, q, s, group, eps, int8 ? -128. : -448., int8 ? 127. : 448., ue8m0, SGLAMD_QUANT_FORM_RECIPROCAL, col,
              silu);
  return std::make_tuple(q, s);
}

// sglang_per_token_quant_fp8 / per_token_quant_int8 for a contiguous device tensor.
optional<std::tuple<Tensor, Tensor>> per_token_quant(const Tensor& x, bool int8) {
  if (any_observed(x)) return {};
  if (x.dim() < 1 || !x.is_cuda() || !x.is_contiguous() || x.numel() == 0) return {};
  const ScalarType t = x.scalar_type();
  if (!(t == at::kFloat || is_half(t)) || (!int8 && (x.dim() != 2 || x.size(1) % 4))) return {};
  const c10::DeviceGuard guard(x.device());
  Tensor q = empty(x.sizes(), int8 ? at::kChar : kFp8, x);
  c10::SmallVector<int64_t, 8> shape(x.sizes().begin(), x.sizes().end());
  shape.back() = 1;
  Tensor s = empty(shape, at::kFloat, x);
  if (int8)
    per_token_quant_int8_(x, q, s);
  else
    sgl_per_token_quant_fp8(x, q, s);
  return std::make_tuple(q, s);
}

// fused_rms_fp8_group_quant (quantization/fused_fp8_quant.py states the contract)
std::tuple<Tensor, Tensor, optional<Tensor>, optional<Tensor>, optional<Tensor>> fused_rms_group_quant(
    const Tensor& x1, const Tensor& w1, double eps1, const optional<Tensor>& x2, const optional<Tensor>& w2,
    optional<double> eps2, const optional<Tensor>& res1, bool want_y1) {
  TORCH_CHECK(x1.dim() == 2 && x1.is_cuda(), "inp1 must be a 2D device tensor");
  const ScalarType t = x1.scalar_type();
  TORCH_CHECK(is_half(t), "inp1 must be Half or BFloat16");
  const int64_t m = x1.size(0), n1 = x1.size(1);
  TORCH_CHECK(x1.stride(1) == 1, "inp1 rows must be contiguous");
  TORCH_CHECK(w1.numel() == n1 && w1.is_contiguous(), "inp1_weight must be contiguous [N1]");
  TORCH_CHECK(w1.scalar_type() == at::kFloat || is_half(w1.scalar_type()), "weights must be Float, Half or BFloat16");
  const c10::DeviceGuard guard(x1.device());
  optional<Tensor> res_out, y1, y2;
  int64_t n2 = 0;
  if (res1) {
    TORCH_CHECK(res1->sizes() == x1.sizes() && res1->scalar_type() == t && res1->is_contiguous(),
                "res1 must match inp1");
    res_out = empty({m, n1}, t, x1);
  }
  if (x2) {
    TORCH_CHECK(x2->dim() == 2 && x2->size(0) == m && x2->scalar_type() == t && x2->stride(1) == 1,
                "inp2 must be [M, N2] in inp1's dtype with contiguous rows");
    TORCH_CHECK(w2.has_value() && eps2.has_value(), "inp2 needs its weight and epsilon");
    n2 = x2->size(1);
    TORCH_CHECK(w2->numel() == n2 && w2->is_contiguous() && w2->scalar_type() == w1.scalar_type(),
                "inp2_weight must be contiguous [N2] in inp1_weight's dtype");
    y2 = empty({m, n2}, t, x1);
  }
  Tensor q = empty({m, n1}, kFp8, x1), s = empty({m, cdiv(n1, 128)}, at::kFloat, x1);
  if (want_y1) y1 = empty({m, n1}, t, x1);
  auto ptr = [](const optional<Tensor>& o) -> void* { return o ? o->data_ptr() : nullptr; };
  check(sglamd_fused_rms_fp8_group_quant(
      x1.data_ptr(), x1.stride(0), w1.data_ptr(), (float)eps1, ptr(res1), m, n1, q.data_ptr(), s.data_ptr<float>(),
      ptr(y1), ptr(res_out), ptr(x2), x2 ? x2->stride(0) : 0, ptr(w2), x2 ? (float)*eps2 : 0.f, n2, ptr(y2), tag(t),
      tag(w1.scalar_type()), 128, stream_of(x1)));
  return {q, s, y1, y2, res_out};
}

// ---------------------------------------------------------------------------------------
// dense GEMMs
// ---------------------------------------------------------------------------------------
// fp32 split-K scratch when the library can use one for this shape; from the caching allocator, so calls on other
// streams and threads have their own.
Tensor gemm_workspace(int64_t m, int64_t n, int64_t k, bool row_scaled, const Tensor& like, void** ptr,
                      int64_t* bytes) {
  *bytes = row_scaled || k % 128 == 0 ? sglamd_gemm_workspace_bytes(m, n, k) : 0;
  *ptr = nullptr;
  if (*bytes <= 0) return Tensor();
  Tensor ws = empty({*bytes}, at::kByte, like);
  *ptr = ws.data_ptr();
  return ws;
}

bool is_contiguous_vector(const Tensor& t) {
  return t.is_contiguous() && (t.dim() == 1 || (t.dim() == 2 && std::min(t.size(0), t.size(1)) == 1));
}

void check_mm_operands(const Tensor& a, const Tensor& b) {
  TORCH_CHECK(a.is_cuda(), "mat_a must be a CUDA tensor");
  TORCH_CHECK(b.is_cuda(), "mat_b must be a CUDA tensor");
  TORCH_CHECK(a.dim() == 2, "mat_a must be a 2D tensor");
  TORCH_CHECK(b.dim() == 2, "mat_b must be a 2D tensor");
  TORCH_CHECK(a.stride(1) == 1, "mat_a must be a row major tensor");
  TORCH_CHECK(b.stride(0) == 1, "mat_b must be a column major tensor");
  TORCH_CHECK(a.size(1) == b.size(0), "mat_a and mat_b shapes cannot be multiplied");
}

void check_fp8_operands(const Tensor& a, const Tensor& b, ScalarType out_dtype) {
  check_mm_operands(a, b);
  TORCH_CHECK((a.size(1) * a.element_size()) % 16 == 0, "mat_a must be multiple of 16 bytes for memory alignment");
  TORCH_CHECK((b.size(0) * b.element_size()) % 16 == 0, "mat_b must be multiple of 16 bytes for memory alignment");
  TORCH_CHECK(a.scalar_type() == kFp8, "mat_a must be Float8_e4m3fn");
  TORCH_CHECK(b.scalar_type() == kFp8, "mat_b must be Float8_e4m3fn");
  TORCH_CHECK(is_half(out_dtype), "out_dtype must be Half or BFloat16");
}

// fp8_blockwise_gemm_kernel.cu:425-522 (checks :431-463)
Tensor fp8_blockwise_scaled_mm(const Tensor& a, const Tensor& b, const Tensor& sa, const Tensor& sb,
                               ScalarType out_dtype) {
  check_fp8_operands(a, b, out_dtype);
  const int64_t m = a.size(0), k = a.size(1), n = b.size(1);
  TORCH_CHECK(sa.dim() == 2 && sb.dim() == 2, "scales must be 2D tensors");
  TORCH_CHECK(m == sa.size(0), "size of scales_a is not matched");
  TORCH_CHECK(k / 128 == sa.size(1), "size of scales_a is not matched");
  TORCH_CHECK(sa.stride(0) == 1 || is_contiguous_vector(sa), "scales_a must be M major");
  TORCH_CHECK(k / 128 == sb.size(0), "size of scales_b is not matched");
  TORCH_CHECK(n / 128 == sb.size(1), "size of scales_b is not matched");
  TORCH_CHECK(sb.stride(0) == 1 || is_contiguous_vector(sb), "scales_b must be K major");
  TORCH_CHECK(sa.scalar_type() == at::kFloat, "scales_a must be Float32");
  TORCH_CHECK(sb.scalar_type() == at::kFloat, "scales_b must be Float32");
  TORCH_CHECK(k % 128 == 0 && n % 128 == 0, "K and N must be multiples of the 128x128 scale block");
  const c10::DeviceGuard guard(a.device());
  Tensor out = empty({m, n}, out_dtype, a);
  if (m == 0) return out;
  void* wp;
  int64_t wb;
  const Tensor ws = gemm_workspace(m, n, k, false, a, &wp, &wb);
  check(sglamd_fp8_blockwise_scaled_mm(a.data_ptr(), ld(a, 0), b.data_ptr(), ld(b, 1), sa.data_ptr<float>(),
                                       sa.stride(0), sa.stride(1), sb.data_ptr<float>(), sb.stride(1), sb.stride(0),
                                       out.data_ptr(), n, tag(out_dtype), m, n, k, wp, wb, stream_of(a)));
  return out;
}

// Row-major operands: a [m, k], b [n, k], sa [m, ceil(k/128)], sb [ceil(n/128), ceil(k/128)], c [m, n] preallocated
// (fp8_kernel.py:1135-1281, int8_kernel.py:355-425).  pow2: every scale is a power of two (expanded UE8M0 scales),
// which lets the large-tile kernel apply them inside the MFMA.
void block_matmul_(const Tensor& a, const Tensor& b, const Tensor& sa, const Tensor& sb, const Tensor& c, bool int8,
                   bool pow2) {
  const int64_t m = a.size(0), k = a.size(1), n = b.size(0);
  if (m == 0) return;
  const c10::DeviceGuard guard(a.device());
  void* wp;
  int64_t wb;
  const Tensor ws = gemm_workspace(m, n, k, false, a, &wp, &wb);
  auto fn = int8 ? sglamd_int8_blockwise_scaled_mm
                 : pow2 ? sglamd_fp8_blockwise_scaled_mm_pow2 : sglamd_fp8_blockwise_scaled_mm;
  check(fn(a.data_ptr(), ld(a, 0), b.data_ptr(), ld(b, 0), (float*)sa.data_ptr(), sa.stride(0), sa.stride(1),
           (float*)sb.data_ptr(), sb.stride(0), sb.stride(1), c.data_ptr(), c.stride(0), tag(c.scalar_type()), m, n, k,
           wp, wb, stream_of(a)));
}

void w8a8_block_fp8_matmul_(const Tensor& a, const Tensor& b, const Tensor& sa, const Tensor& sb, const Tensor& c,
                            bool pow2_scales) {
  block_matmul_(a, b, sa, sb, c, false, pow2_scales);
}

void w8a8_block_int8_matmul_(const Tensor& a, const Tensor& b, const Tensor& sa, const Tensor& sb, const Tensor& c) {
  block_matmul_(a, b, sa, sb, c, true, false);
}

// The block-scaled GEMM with a general scale-block shape (fp8_kernel.py:780-869, int8_kernel.py:228-441): block_n and
// block_k in {64, 128}.
void block_scaled_mm_any_(const Tensor& a, const Tensor& b, const Tensor& sa, const Tensor& sb, const Tensor& c,
                          int64_t block_n, int64_t block_k) {
  const int64_t m = a.size(0), k = a.size(1), n = b.size(0);
  if (m == 0) return;
  TORCH_CHECK((a.scalar_type() == kFp8 || a.scalar_type() == at::kChar) && b.scalar_type() == a.scalar_type(),
              "A and B must both be Float8_e4m3fn or both Int8");
  const c10::DeviceGuard guard(a.device());
  check(sglamd_block_scaled_mm_any(a.data_ptr(), ld(a, 0), b.data_ptr(), ld(b, 0), (float*)sa.data_ptr(), sa.stride(0),
                                   sa.stride(1), (float*)sb.data_ptr(), sb.stride(0), sb.stride(1), c.data_ptr(),
                                   c.stride(0), tag(c.scalar_type()), tag(a.scalar_type()), m, n, k, (int)block_n,
                                   (int)block_k, stream_of(a)));
}

Tensor rowwise_mm(bool int8, const Tensor& a, const Tensor& b, const Tensor& sa, const Tensor& sb, ScalarType out_dtype,
                  const optional<Tensor>& bias) {
  const int64_t m = a.size(0), k = a.size(1), n = b.size(1);
  TORCH_CHECK(sa.numel() == m, "size of scales_a is not matched");
  TORCH_CHECK(sb.numel() == n, "size of scales_b is not matched");
  TORCH_CHECK(sa.is_contiguous(), "scales_a must be contiguous");
  TORCH_CHECK(sb.is_contiguous(), "scales_b msut be contiguous");
  TORCH_CHECK(sa.scalar_type() == at::kFloat, "scales_a must be Float32");
  TORCH_CHECK(sb.scalar_type() == at::kFloat, "scales_b must be Float32");
  if (bias) {
    TORCH_CHECK(bias->numel() == n, "size of bias is not matched");
    TORCH_CHECK(bias->is_contiguous(), "bias must be contiguous");
    TORCH_CHECK(bias->scalar_type() == out_dtype, "bias dtype must match output dtype");
  }
  const c10::DeviceGuard guard(a.device());
  Tensor out = empty({m, n}, out_dtype, a);
  if (m == 0) return out;
  void* wp;
  int64_t wb;
  const Tensor ws = gemm_workspace(m, n, k, true, a, &wp, &wb);
  auto fn = int8 ? sglamd_int8_scaled_mm : sglamd_fp8_scaled_mm;
  check(fn(a.data_ptr(), ld(a, 0), b.data_ptr(), ld(b, 1), sa.data_ptr<float>(), sb.data_ptr<float>(),
           bias ? bias->data_ptr() : nullptr, out.data_ptr(), n, tag(out_dtype), m, n, k, wp, wb, stream_of(a)));
  return out;
}

// fp8_gemm_kernel.cu:1095-1173 (checks :1102-1132)
Tensor fp8_scaled_mm(const Tensor& a, const Tensor& b, const Tensor& sa, const Tensor& sb, ScalarType out_dtype,
                     const optional<Tensor>& bias) {
  check_fp8_operands(a, b, out_dtype);
  TORCH_CHECK((b.size(1) * 2) % 16 == 0, "out must be multiple of 16 bytes for memory alignment");
  return rowwise_mm(false, a, b, sa, sb, out_dtype, bias);
}

// int8_gemm_kernel.cu:663-747 (checks :670-695)
Tensor int8_scaled_mm(const Tensor& a, const Tensor& b, const Tensor& sa, const Tensor& sb, ScalarType out_dtype,
                      const optional<Tensor>& bias) {
  check_mm_operands(a, b);
  TORCH_CHECK(a.size(1) % 16 == 0, "mat_a.size(1) must be multiple of 16 for memory alignment");
  TORCH_CHECK(b.size(0) % 16 == 0, "mat_b.size(0) must be multiple of 16 for memory alignment");
  TORCH_CHECK(b.size(1) % 8 == 0, "mat_b.size(1) must be multiple of 8 for memory alignment");
  TORCH_CHECK(a.scalar_type() == at::kChar, "mat_a must be Int8");
  TORCH_CHECK(b.scalar_type() == at::kChar, "mat_b must be Int8");
  TORCH_CHECK(is_half(out_dtype), "out_dtype must be Half or BFloat16");
  return rowwise_mm(true, a, b, sa, sb, out_dtype, bias);
}

bool plain_weight(const Tensor& w, const Tensor& x, ScalarType t) {
  return w.dim() == 2 && w.is_cuda() && w.device() == x.device() && w.scalar_type() == t && w.is_contiguous() &&
         w.size(0) > 0;
}

// float [ceil(n/128), ceil(k/128)] scales, or the int32 words of packed UE8M0 exponents, one row of words per weight
// row
bool plain_block_scale(const Tensor& ws, const Tensor& w) {
  const int64_t n = w.size(0), kb = cdiv(w.size(1), 128);
  if (ws.dim() != 2 || ws.device() != w.device()) return false;
  if (ws.scalar_type() == at::kFloat) return ws.size(0) == cdiv(n, 128) && ws.size(1) == kb;
  return ws.scalar_type() == at::kInt && ws.size(0) == n && ws.size(1) == cdiv(kb, 4);
}

bool plain_bias(const optional<Tensor>& bias, const Tensor& out_like, int64_t n, ScalarType t) {
  return !bias || (bias->dim() == 1 && bias->numel() == n && bias->is_contiguous() && bias->scalar_type() == t &&
                   bias->device() == out_like.device());
}

// Whether a bias goes into the block-scaled GEMM.  The large-tile persistent kernel reads it in aligned words; with any
// other bias that launch would run one tile per workgroup instead, which is slower and sums in another order, so there
// the bias is added behind the GEMM and the result is the same wherever the bias lies.
bool bias_in_gemm(const optional<Tensor>& bias, int64_t n) {
  return bias && ((uintptr_t)bias->data_ptr() & 3) == 0 && n >= 32;
}

// The block-scaled linear layer (fp8_utils.py:612-642,645-696,814-834): quantise x [m, k] per 1x128 group, multiply by
// weight [n, k] with 128x128 block scales, add the bias.
optional<Tensor> block_linear(const Tensor& x, const Tensor& w, const Tensor& ws, const optional<Tensor>& bias) {
  if (any_observed(x, w, ws, bias)) return {};
  const ScalarType t = x.scalar_type();
  if (x.dim() != 2 || !x.is_cuda() || !is_half(t) || !x.is_contiguous() || x.size(0) == 0) return {};
  if (!plain_weight(w, x, kFp8) || w.size(1) != x.size(1) || !plain_block_scale(ws, w)) return {};
  const int64_t m = x.size(0), k = x.size(1), n = w.size(0), kb = k / 128;
  if (k == 0 || k % 128 || !plain_bias(bias, x, n, t)) return {};
  const bool ue8m0 = ws.scalar_type() == at::kInt;
  const c10::DeviceGuard guard(x.device());
  Tensor out = empty({m, n}, t, x);
  Scratch sc;
  const int64_t q = sc.take(m * k), sa = sc.take(4 * m * kb), sb = ue8m0 ? sc.take(4 * cdiv(n, 128) * kb) : 0;
  const int64_t wb = sglamd_gemm_workspace_bytes(m, n, k), wp = sc.take(wb > 0 ? wb : 0);
  sc.allocate(x);
  void* st = stream_of(x);
  if (!ue8m0) {
    const bool inside = bias_in_gemm(bias, n);
    check(sglamd_fp8_block_linear(x.data_ptr(), tag(t), m, k, w.data_ptr(), k, ws.data_ptr<float>(), ws.stride(0), ws.stride(1),
                                  inside ? bias->data_ptr() : nullptr, out.data_ptr(), n, n, sc.at(q), (float*)sc.at(sa),
                                  wb > 0 ? sc.at(wp) : nullptr, wb, st));
    if (bias && !inside) out.add_(*bias);
    return out;
  }
  check(sglamd_ue8m0_linear_operands(x.data_ptr(), tag(t), sc.at(q), (float*)sc.at(sa), m, k, ws.data_ptr(), ws.stride(0),
                                     ws.stride(1), (float*)sc.at(sb), cdiv(n, 128), st));
  const float* wsp = (const float*)sc.at(sb);
  const int64_t ws_n = kb, ws_k = 1;
  if (bias_in_gemm(bias, n)) {
    check(sglamd_fp8_blockwise_scaled_mm_bias(sc.at(q), k, w.data_ptr(), k, (float*)sc.at(sa), 1, m, wsp, ws_n, ws_k, ue8m0,
                                              bias->data_ptr(), out.data_ptr(), n, tag(t), m, n, k,
                                              wb > 0 ? sc.at(wp) : nullptr, wb, st));
    return out;
  }
  check(sglamd_fp8_blockwise_scaled_mm_pow2(sc.at(q), k, w.data_ptr(), k, (float*)sc.at(sa), 1, m, wsp, ws_n, ws_k, out.data_ptr(), n, tag(t), m, n, k,
           wb > 0 ? sc.at(wp) : nullptr, wb, st));
  if (bias) out.add_(*bias);
  return out;
}

// The block matmul of operands that are quantised already (w8a8_block_fp8_matmul, w8a8_block_int8_matmul), float
// scales, [m, k] x [n, k]; with an optional bias for the linear layers that take quantised inputs.
optional<Tensor> block_matmul(const Tensor& a, const Tensor& b, const Tensor& sa, const Tensor& sb, ScalarType out_dtype,
                              const optional<Tensor>& bias) {
  if (any_observed(a, b, sa, sb, bias)) return {};
  const ScalarType t = a.scalar_type();
  if (a.dim() != 2 || !a.is_cuda() || (t != kFp8 && t != at::kChar) || !a.is_contiguous() || a.size(0) == 0) return {};
  if (!plain_weight(b, a, t) || b.size(1) != a.size(1) || !is_half(out_dtype)) return {};
  const int64_t m = a.size(0), k = a.size(1), n = b.size(0), kb = cdiv(k, 128);
  if (sa.dim() != 2 || sa.scalar_type() != at::kFloat || sa.device() != a.device() || sa.size(0) != m ||
      sa.size(1) != kb || sb.scalar_type() != at::kFloat || !plain_block_scale(sb, b) ||
      !plain_bias(bias, a, n, out_dtype))
    return {};
  const c10::DeviceGuard guard(a.device());
  Tensor out = empty({m, n}, out_dtype, a);
  if (t == kFp8 && bias_in_gemm(bias, n)) {
    void* wp;
    int64_t wb;
    const Tensor ws = gemm_workspace(m, n, k, false, a, &wp, &wb);
    check(sglamd_fp8_blockwise_scaled_mm_bias(a.data_ptr(), k, b.data_ptr(), k, sa.data_ptr<float>(), sa.stride(0),
                                              sa.stride(1), sb.data_ptr<float>(), sb.stride(0), sb.stride(1), 0,
                                              bias->data_ptr(), out.data_ptr(), n, tag(out_dtype), m, n, k, wp, wb,
                                              stream_of(a)));
    return out;
  }
  block_matmul_(a, b, sa, sb, out, t == at::kChar, false);
  if (bias) out.add_(*bias);
  return out;
}

// The per-channel FP8 linear layer with per-token activation scales (fp8_utils.py:1458-1560): weight is the [k, n]
// view of the [n, k] parameter, weight_scale one value per output column.
optional<Tensor> row_linear(const Tensor& x, const Tensor& weight, const Tensor& ws, const optional<Tensor>& bias) {
  if (any_observed(x, weight, ws, bias)) return {};
  const ScalarType t = x.scalar_type();
  if (x.dim() != 2 || !x.is_cuda() || !is_half(t) || !x.is_contiguous() || x.size(0) == 0) return {};
  if (weight.dim() != 2 || weight.device() != x.device() || weight.scalar_type() != kFp8 || weight.stride(0) != 1)
    return {};
  const int64_t m = x.size(0), k = x.size(1), n = weight.size(1);
  if (weight.size(0) != k || k == 0 || k % 16 || n == 0 || n % 8 || ws.numel() != n || ws.scalar_type() != at::kFloat ||
      !ws.is_contiguous() || ws.device() != x.device() || !plain_bias(bias, x, n, t))
    return {};
  const c10::DeviceGuard guard(x.device());
  Tensor out = empty({m, n}, t, x);
  Scratch sc;
  const int64_t q = sc.take(m * k), sa = sc.take(4 * m);
  const int64_t wb = sglamd_gemm_workspace_bytes(m, n, k), wp = sc.take(wb > 0 ? wb : 0);
  sc.allocate(x);
  void* st = stream_of(x);
  check(sglamd_fp8_row_linear(x.data_ptr(), tag(t), m, k, weight.data_ptr(), ld(weight, 1), ws.data_ptr<float>(),
                              bias ? bias->data_ptr() : nullptr, out.data_ptr(), n, n, sc.at(q), (float*)sc.at(sa),
                              wb > 0 ? sc.at(wp) : nullptr, wb, st));
  return out;
}

// ---------------------------------------------------------------------------------------
// MoE
// ---------------------------------------------------------------------------------------
void check_router(const Tensor& weights, const Tensor& ids, const Tensor& gating, const optional<Tensor>& bias) {
  const ScalarType t = gating.scalar_type();
  TORCH_CHECK(t == at::kFloat || is_half(t), "gating_output must be float32, float16, or bfloat16");
  TORCH_CHECK(gating.dim() == 2, "gating_output must be 2D tensor [num_tokens, num_experts]");
  TORCH_CHECK(weights.dim() == 2, "topk_weights must be 2D tensor [num_tokens, topk]");
  TORCH_CHECK(ids.dim() == 2, "topk_indices must be 2D tensor [num_tokens, topk]");
  TORCH_CHECK(gating.size(0) == weights.size(0),
              "First dimension of topk_weights must match num_tokens in gating_output");
  TORCH_CHECK(gating.size(0) == ids.size(0), "First dimension of topk_indices must match num_tokens in gating_output");
  TORCH_CHECK(weights.size(-1) == ids.size(-1), "Second dimension of topk_indices must match topk in topk_weights");
  TORCH_CHECK(weights.size(-1) <= gating.size(-1), "topk must be less than or equal to num_experts");
  TORCH_CHECK(weights.scalar_type() == at::kFloat && ids.scalar_type() == at::kInt,
              "topk_weights must be Float and topk_indices Int");
  check_input(weights, "topk_weights");
  check_input(ids, "topk_indices");
  check_input(gating, "gating_output");
  if (bias) {
    TORCH_CHECK(bias->dim() == 1, "correction_bias must be 1D tensor [num_experts]");
    TORCH_CHECK(bias->size(0) == gating.size(-1), "correction_bias size must match num_experts");
    TORCH_CHECK(bias->scalar_type() == at::kFloat, "correction_bias must be float32, got ", bias->scalar_type());
    check_input(*bias, "correction_bias");
  }
}

// moe_topk_softmax_kernels.cu:718-810 (checks :726-775)
void topk_softmax(const Tensor& weights, const Tensor& ids, const Tensor& gating, bool renormalize, double softcapping,
                  const optional<Tensor>& bias) {
  check_router(weights, ids, gating, bias);
  if (gating.size(0) == 0) return;
  const c10::DeviceGuard guard(gating.device());
  check(sglamd_topk_softmax(weights.data_ptr<float>(), ids.data_ptr<int32_t>(), gating.data_ptr(),
                            tag(gating.scalar_type()), gating.size(0), gating.size(1), weights.size(-1), renormalize,
                            (float)softcapping, bias ? bias->data_ptr<float>() : nullptr, stream_of(gating)));
}

// moe_topk_sigmoid_kernels.cu:496-600 (checks :503-548)
void topk_sigmoid(const Tensor& weights, const Tensor& ids, const Tensor& gating, bool renormalize,
                  const optional<Tensor>& bias) {
  check_router(weights, ids, gating, bias);
  if (gating.size(0) == 0) return;
  const c10::DeviceGuard guard(gating.device());
  check(sglamd_topk_sigmoid(weights.data_ptr<float>(), ids.data_ptr<int32_t>(), gating.data_ptr(),
                            tag(gating.scalar_type()), gating.size(0), gating.size(1), weights.size(-1), renormalize,
                            bias ? bias->data_ptr<float>() : nullptr, stream_of(gating)));
}

// moe_align_kernel.cu:317-383.  Sizes of the outputs are the caller's responsibility there; here the ones that would
// make the kernel write out of bounds are checked.
void moe_align_block_size(const Tensor& ids, int64_t num_experts, int64_t block_size, const Tensor& sorted,
                          const Tensor& experts, const Tensor& post_pad, const Tensor& cumsum, bool pad_sorted) {
  TORCH_CHECK(ids.is_cuda() && ids.is_contiguous(), "topk_ids must be a contiguous CUDA tensor");
  TORCH_CHECK(ids.scalar_type() == at::kInt || ids.scalar_type() == at::kLong,
              "topk_ids must be an integral tensor (int32/int64)");
  auto i32 = [](const Tensor& t, const char* name) {
    TORCH_CHECK(t.is_cuda() && t.is_contiguous() && t.scalar_type() == at::kInt, name,
                " must be a contiguous int32 CUDA tensor");
  };
  i32(sorted, "sorted_token_ids");
  i32(experts, "experts_ids");
  i32(post_pad, "num_tokens_post_pad");
  i32(cumsum, "cumsum_buffer");
  const int64_t numel = ids.numel(), max_padded = sorted.size(0);
  const int64_t worst = numel + std::min(numel, num_experts) * (block_size - 1);
  TORCH_CHECK(max_padded >= std::min(worst, numel * block_size), "sorted_token_ids is too small for the padded spans");
  TORCH_CHECK(experts.numel() * block_size >= max_padded - block_size + 1, "experts_ids is too small");
  TORCH_CHECK(cumsum.numel() >= num_experts + 1, "cumsum_buffer must hold num_experts + 1 entries");
  const c10::DeviceGuard guard(ids.device());
  check(sglamd_moe_align_block_size(ids.data_ptr(), tag(ids.scalar_type()), numel, (int)num_experts, (int)block_size,
                                    sorted.data_ptr<int32_t>(), max_padded, experts.data_ptr<int32_t>(),
                                    post_pad.data_ptr<int32_t>(), cumsum.data_ptr<int32_t>(), pad_sorted,
                                    stream_of(ids)));
}

void act_and_mul(const char* name, int (*fn)(const void*, void*, int, int64_t, int64_t, void*), const Tensor& out,
                 const Tensor& input) {
  check_input(input, "input");
  check_input(out, "out");
  TORCH_CHECK(is_half(input.scalar_type()) && out.scalar_type() == input.scalar_type(), name,
              " takes Half or BFloat16 tensors of one dtype");
  const int64_t d = input.size(-1) / 2, rows = input.numel() ? input.numel() / input.size(-1) : 0;
  TORCH_CHECK(out.numel() == rows * d, "out has the wrong number of elements");
  const c10::DeviceGuard guard(input.device());
  check(fn(input.data_ptr(), out.data_ptr(), tag(input.scalar_type()), rows, d, stream_of(input)));
}

// elementwise/activation.cu:82-149
void silu_and_mul(const Tensor& out, const Tensor& input) {
  act_and_mul("silu_and_mul", sglamd_silu_and_mul, out, input);
}
void gelu_tanh_and_mul(const Tensor& out, const Tensor& input) {
  act_and_mul("gelu_tanh_and_mul", sglamd_gelu_tanh_and_mul, out, input);
}
void gelu_and_mul(const Tensor& out, const Tensor& input) {
  act_and_mul("gelu_and_mul", sglamd_gelu_and_mul, out, input);
}

// common_extension.cc:180-181: input [tokens, topk, hidden] -> output [tokens, hidden]
void moe_sum_reduce(const Tensor& input, const Tensor& output, double routed_scaling_factor) {
  check_input(input, "input");
  check_input(output, "output");
  TORCH_CHECK(input.dim() == 3 && output.dim() == 2, "input must be 3D and output 2D");
  const int64_t tokens = input.size(0), topk = input.size(1), d = input.size(2);
  TORCH_CHECK(output.size(0) == tokens && output.size(1) == d, "output shape does not match input");
  TORCH_CHECK(is_half(input.scalar_type()) && output.scalar_type() == input.scalar_type(),
              "moe_sum_reduce takes Half or BFloat16 tensors of one dtype");
  const c10::DeviceGuard guard(input.device());
  check(sglamd_moe_sum_reduce(input.data_ptr(), output.data_ptr(), tag(input.scalar_type()), tokens, (int)topk, d,
                              (float)routed_scaling_factor, stream_of(input)));
}

// prepare_moe_input.cu:130-156 (dtype check :141)
void prepare_moe_input(const Tensor& ids, const Tensor& offsets, const optional<Tensor>& blockscale_offsets,
                       const Tensor& sizes1, const Tensor& sizes2, const Tensor& input_perm, const Tensor& output_perm,
                       int64_t num_experts, int64_t n, int64_t k) {
  TORCH_CHECK(ids.scalar_type() == at::kInt, "topk_ids must be int32");
  check_input(ids, "topk_ids");
  const int64_t numel = ids.numel(), topk = ids.dim() == 2 ? ids.size(1) : 1;
  auto i32 = [](const Tensor& t, const char* name, int64_t need) {
    check_input(t, name);
    TORCH_CHECK(t.scalar_type() == at::kInt && t.numel() >= need, name, " must be int32 with at least ", need,
                " elements");
  };
  i32(offsets, "expert_offsets", num_experts + 1);
  i32(sizes1, "problem_sizes1", num_experts * 3);
  i32(sizes2, "problem_sizes2", num_experts * 3);
  i32(input_perm, "input_permutation", numel);
  i32(output_perm, "output_permutation", numel);
  if (blockscale_offsets) {
    check_input(*blockscale_offsets, "blockscale_offsets");
    TORCH_CHECK(blockscale_offsets->scalar_type() == at::kInt && blockscale_offsets->numel() >= num_experts + 1,
                "blockscale_offsets must be int32 with num_experts + 1 elements");
  }
  const c10::DeviceGuard guard(ids.device());
  check(sglamd_prepare_moe_input(ids.data_ptr<int32_t>(), numel, (int)topk, (int)num_experts, n, k,
                                 offsets.data_ptr<int32_t>(),
                                 blockscale_offsets ? blockscale_offsets->data_ptr<int32_t>() : nullptr,
                                 sizes1.data_ptr<int32_t>(), sizes2.data_ptr<int32_t>(), input_perm.data_ptr<int32_t>(),
                                 output_perm.data_ptr<int32_t>(), stream_of(ids)));
}

// prepare_moe_input.cu:213-246 (same-dtype check :215-217; float32, half, bfloat16, fp8 and uint8 rows)
void shuffle_rows(const Tensor& input, const Tensor& map, const Tensor& output) {
  const ScalarType t = input.scalar_type();
  TORCH_CHECK(t == output.scalar_type(), "Input and output tensors must have the same data type");
  TORCH_CHECK(is_half(t) || t == at::kFloat || t == kFp8 || t == at::kByte,
              "[moe replicate input] data type dispatch fail!");
  check_input(input, "input");
  check_input(output, "output");
  check_input(map, "dst2src_map");
  TORCH_CHECK(map.scalar_type() == at::kInt && map.numel() >= output.size(0),
              "dst2src_map must be int32 with one entry per output row");
  TORCH_CHECK(input.dim() == 2 && output.dim() == 2 && input.size(1) == output.size(1),
              "input and output must be 2D with the same number of columns");
  const c10::DeviceGuard guard(input.device());
  check(sglamd_shuffle_rows(input.data_ptr(), map.data_ptr<int32_t>(), output.data_ptr(), output.size(0),
                            input.size(1) * input.element_size(), stream_of(input)));
}

// prepare_moe_input.cu:300-376 (checks :306-327)
void apply_shuffle_mul_sum(const Tensor& input, const Tensor& output, const Tensor& perm,
                           const optional<Tensor>& factors) {
  TORCH_CHECK(input.dim() == 2, "input_tensor must be 2D [m * topk, row_stride]");
  TORCH_CHECK(output.dim() == 2, "output_tensor must be 2D [m, row_stride]");
  TORCH_CHECK(perm.dim() == 1, "permutation must be 1D [m * topk]");
  const int64_t m = output.size(0), row_stride = output.size(1), topk = m ? perm.size(0) / m : 1;
  TORCH_CHECK(perm.size(0) == m * topk, "permutation size must match m * topk");
  TORCH_CHECK(perm.scalar_type() == at::kInt, "permutation must be int32");
  TORCH_CHECK(is_half(output.scalar_type()) && input.scalar_type() == output.scalar_type(),
              "input and output must both be Half or BFloat16");
  TORCH_CHECK(input.size(1) == row_stride && input.size(0) >= m * topk, "input shape does not match output");
  check_input(input, "input");
  check_input(output, "output");
  check_input(perm, "permutation");
  if (factors) {
    TORCH_CHECK(factors->scalar_type() == output.scalar_type(), "Factors must match output dtype");
    TORCH_CHECK(factors->numel() == m * topk, "Factors must have shape [m * topk]");
    check_input(*factors, "factors");
  }
  if (m == 0) return;
  const c10::DeviceGuard guard(input.device());
  check(sglamd_apply_shuffle_mul_sum(input.data_ptr(), output.data_ptr(), perm.data_ptr<int32_t>(),
                                     factors ? factors->data_ptr() : nullptr, tag(output.scalar_type()), m, (int)topk,
                                     row_stride, stream_of(input)));
}

// fp8_blockwise_moe_kernel.cu:650-810 (checks :669-707).  The pointer, stride and layout containers are scratch of the
// reference's CUTLASS launch; they are checked like the reference checks them and otherwise unused.  `b` is the
// [E, K, N] column-major view of contiguous [E, N, K] weights, `scales_b` the [E, K/128, N/128] view of contiguous
// [E, N/128, K/128] scales.  The sorted-block schedule is built in `workspace` when it is large enough, else in a
// buffer from torch's caching allocator.
void fp8_blockwise_scaled_grouped_mm(const Tensor& output, const Tensor&, const Tensor&, const Tensor&, const Tensor&,
                                     const Tensor&, const Tensor& a, const Tensor& b, const Tensor& scales_a,
                                     const Tensor& scales_b, const Tensor& stride_a, const Tensor& stride_b,
                                     const Tensor& stride_c, const Tensor& layout_sfa, const Tensor& layout_sfb,
                                     const Tensor& problem_sizes, const Tensor& expert_offsets,
                                     const Tensor& workspace) {
  TORCH_CHECK(problem_sizes.dim() == 2, "problem_sizes must be 2D tensor");
  TORCH_CHECK(problem_sizes.size(1) == 3, "problem_sizes must have shape (num_experts, 3)");
  TORCH_CHECK(problem_sizes.size(0) == expert_offsets.size(0),
              "Number of experts in problem_sizes must match expert_offsets");
  TORCH_CHECK(problem_sizes.scalar_type() == at::kInt, "problem_sizes must be int32");
  TORCH_CHECK(a.scalar_type() == kFp8, "a must be kFloat8_e4m3fn");
  TORCH_CHECK(b.scalar_type() == kFp8, "b must be kFloat8_e4m3fn");
  TORCH_CHECK(is_half(output.scalar_type()), "output must be bfloat16 or half");
  TORCH_CHECK(scales_a.scalar_type() == at::kFloat, "scales_a must be float32");
  TORCH_CHECK(scales_b.scalar_type() == at::kFloat, "scales_b must be float32");
  TORCH_CHECK(stride_a.scalar_type() == at::kLong, "stride_a must be int64");
  TORCH_CHECK(stride_b.scalar_type() == at::kLong, "stride_b must be int64");
  TORCH_CHECK(stride_c.scalar_type() == at::kLong, "stride_c must be int64");
  TORCH_CHECK(layout_sfa.scalar_type() == at::kInt, "layout_sfa must be int32");
  TORCH_CHECK(layout_sfb.scalar_type() == at::kInt, "layout_sfb must be int32");
  TORCH_CHECK(expert_offsets.scalar_type() == at::kInt, "expert_offsets must be int32");
  TORCH_CHECK(output.dim() == 2, "output must be 2D tensor");
  TORCH_CHECK(a.dim() == 2, "a must be 2D tensor");
  TORCH_CHECK(b.dim() == 3, "b must be 3D tensor");
  TORCH_CHECK(scales_a.dim() == 2, "scales_a must be 2D tensor");
  TORCH_CHECK(scales_b.dim() == 3, "scales_b must be 3D tensor");
  TORCH_CHECK(stride_a.dim() == 1 && stride_b.dim() == 1 && stride_c.dim() == 1, "strides must be 1D tensors");
  TORCH_CHECK(expert_offsets.dim() == 1, "expert_offsets must be 1D tensor");
  TORCH_CHECK(workspace.dim() == 1, "workspace must be 1D tensor");
  const int64_t e = b.size(0), k = b.size(1), n = b.size(2), rows = a.size(0);
  TORCH_CHECK(a.size(1) == k && a.is_contiguous(), "a must be contiguous [rows, K]");
  TORCH_CHECK(b.stride(1) == 1 && b.stride(2) == k && (e == 1 || b.stride(0) == n * k),
              "b must be the [E, K, N] view of contiguous [E, N, K] weights");
  TORCH_CHECK(scales_a.size(0) == rows && scales_a.size(1) == k / 128 && scales_a.is_contiguous(),
              "scales_a must be contiguous [rows, K / 128]");
  TORCH_CHECK(scales_b.size(0) == e && scales_b.size(1) == k / 128 && scales_b.size(2) == n / 128 &&
                  scales_b.stride(1) == 1 && scales_b.stride(2) == k / 128,
              "scales_b must be the [E, K/128, N/128] view of [E, N/128, K/128]");
  TORCH_CHECK(output.size(0) == rows && output.size(1) == n && output.is_contiguous(),
              "output must be contiguous [rows, N]");
  TORCH_CHECK(problem_sizes.size(0) == e, "problem_sizes must have one row per expert");
  check_input(problem_sizes, "problem_sizes");
  TORCH_CHECK(expert_offsets.stride(0) == 1, "expert_offsets must be contiguous");
  if (rows == 0) return;
  const c10::DeviceGuard guard(a.device());
  const int64_t need = sglamd_grouped_mm_workspace_bytes(rows, (int)e);
  Tensor ws = workspace;
  if (!ws.is_cuda() || ws.numel() * ws.element_size() < need || (uintptr_t)ws.data_ptr() % 16 || !ws.is_contiguous())
    ws = empty({need}, at::kByte, a);
  check(sglamd_fp8_blockwise_scaled_grouped_mm(output.data_ptr(), tag(output.scalar_type()), a.data_ptr(), b.data_ptr(),
                                               scales_a.data_ptr<float>(), scales_b.data_ptr<float>(),
                                               problem_sizes.data_ptr<int32_t>(), expert_offsets.data_ptr<int32_t>(),
                                               (int)e, rows, n, k, ws.data_ptr(), ws.numel() * ws.element_size(),
                                               stream_of(a)));
}

// The "expert specialisation" launch of the same grouped GEMM (schema common_extension.cc:483-487; called in place of
// fp8_blockwise_scaled_grouped_mm at python/sglang/srt/layers/moe/cutlass_moe.py:224-237,290-303 with the same operands
// and without the pointer / layout scratch).  Same arithmetic, one implementation here.
void es_fp8_blockwise_scaled_grouped_mm(const Tensor& output, const Tensor& a, const Tensor& b, const Tensor& scales_a,
                                        const Tensor& scales_b, const Tensor& stride_a, const Tensor& stride_b,
                                        const Tensor& stride_d, const Tensor& problem_sizes,
                                        const Tensor& expert_offsets, const Tensor& workspace) {
  const Tensor none = empty({0}, at::kInt, a);
  fp8_blockwise_scaled_grouped_mm(output, none, none, none, none, none, a, b, scales_a, scales_b, stride_a, stride_b,
                                  stride_d, none, none, problem_sizes, expert_offsets, workspace);
}

// The sorted-block grouped GEMM of the block [128, 128] configurations (invoke_fused_moe_kernel,
// fused_moe_triton_kernels.py:702-930).  A e4m3fn or int8 [rows, K] quantised activations with scales A_scale
// [rows, ceil(K/128)]; B of the same type [E, N, K]; B_scale [E, ceil(N/128), ceil(K/128)]; C [num_valid, N] where
// num_valid = topk_ids.numel().
void fused_moe_block_fp8_gemm_(const Tensor& a, const Tensor& a_scale, const Tensor& b, const Tensor& b_scale,
                               const Tensor& c, const optional<Tensor>& topk_weights, const Tensor& sorted,
                               const Tensor& experts, const Tensor& post_pad, bool mul_routed_weight, int64_t top_k,
                               int64_t block_m) {
  const int64_t n = b.size(1), k = b.size(2);
  check_positive(n, "N");
  check_positive(block_m, "block_m");
  const int64_t num_valid = c.numel() / n;
  const bool int8 = a.scalar_type() == at::kChar;
  TORCH_CHECK((int8 || a.scalar_type() == kFp8) && b.scalar_type() == a.scalar_type(),
              "A and B must both be Float8_e4m3fn or both Int8");
  TORCH_CHECK(a.stride(-1) == 1 && b.stride(-1) == 1 && c.is_contiguous(), "A, B rows and C must be contiguous");
  TORCH_CHECK(a_scale.scalar_type() == at::kFloat && b_scale.scalar_type() == at::kFloat, "scales must be Float32");
  TORCH_CHECK(a_scale.size(-1) == cdiv(k, 128) && b_scale.size(-1) == cdiv(k, 128) && b_scale.size(-2) == cdiv(n, 128),
              "scale shapes do not match the 128x128 blocks");
  const int64_t max_blocks = cdiv(sorted.numel(), block_m);
  TORCH_CHECK(experts.numel() >= max_blocks, "expert_ids is too small");
  const c10::DeviceGuard guard(a.device());
  auto fn = int8 ? sglamd_fused_moe_block_int8_gemm : sglamd_fused_moe_block_fp8_gemm;
  check(fn(a.data_ptr(), a.stride(0), a_scale.data_ptr<float>(), a_scale.stride(0), a_scale.stride(1), b.data_ptr(),
           b.stride(0), b.stride(1), b_scale.data_ptr<float>(), b_scale.stride(0), b_scale.stride(1), b_scale.stride(2),
           c.data_ptr(), n, tag(c.scalar_type()), sorted.data_ptr<int32_t>(), experts.data_ptr<int32_t>(),
           post_pad.data_ptr<int32_t>(), topk_weights ? topk_weights->data_ptr<float>() : nullptr, num_valid, (int)top_k,
           mul_routed_weight, (int)block_m, max_blocks, n, k, stream_of(a)));
}

// The sorted-block grouped GEMM beyond block [128, 128]: scale blocks of 64 or 128 (block_n, block_k; A_scale [rows,
// ceil(K/block_k)], B_scale [E, ceil(N/block_n), ceil(K/block_k)]), or both 0 for row scaling: A_scale one value per
// activation row (or a single value: per tensor), B_scale [E, N] per channel (or [E]: per expert).  bias: optional
// [E, N] in C's dtype.
void fused_moe_gemm_any_(const Tensor& a, const Tensor& a_scale, const Tensor& b, const Tensor& b_scale, const Tensor& c,
                         const optional<Tensor>& topk_weights, const Tensor& sorted, const Tensor& experts,
                         const Tensor& post_pad, bool mul_routed_weight, int64_t top_k, int64_t block_m,
                         const optional<std::vector<int64_t>>& block_shape, const optional<Tensor>& bias) {
  const int64_t e = b.size(0), n = b.size(1), k = b.size(2);
  check_positive(n, "N");
  check_positive(block_m, "block_m");
  const int64_t num_valid = c.numel() / n;
  TORCH_CHECK((a.scalar_type() == kFp8 || a.scalar_type() == at::kChar) && b.scalar_type() == a.scalar_type(),
              "A and B must both be Float8_e4m3fn or both Int8");
  TORCH_CHECK(a.stride(-1) == 1 && b.stride(-1) == 1 && c.is_contiguous(), "A, B rows and C must be contiguous");
  TORCH_CHECK(a_scale.scalar_type() == at::kFloat && b_scale.scalar_type() == at::kFloat, "scales must be Float32");
  Tensor as = a_scale, bs = b_scale;
  int64_t bn = 0, bk = 0, a_m, a_k, b_e, b_n, b_k;
  if (block_shape) {
    TORCH_CHECK(block_shape->size() == 2, "block_shape must be [block_n, block_k]");
    bn = (*block_shape)[0], bk = (*block_shape)[1];
    check_positive(bn, "block_n");
    check_positive(bk, "block_k");
    TORCH_CHECK(as.size(-1) == cdiv(k, bk) && bs.size(-1) == cdiv(k, bk) && bs.size(-2) == cdiv(n, bn),
                "scale shapes do not match the scale blocks");
    a_m = as.stride(0), a_k = as.stride(1);
    b_e = bs.stride(0), b_n = bs.stride(1), b_k = bs.stride(2);
  } else {
    TORCH_CHECK(as.numel() == 1 || as.numel() == a.size(0), "the activation scale must be per tensor or per row");
    TORCH_CHECK(bs.numel() == e || bs.numel() == e * n, "the weight scale must be per expert or per channel");
    a_m = as.numel() == 1 ? 0 : 1, a_k = 0;
    b_e = bs.numel() == e ? 1 : n, b_n = bs.numel() == e ? 0 : 1, b_k = 0;
    as = as.contiguous(), bs = bs.contiguous();
  }
  if (bias) {
    TORCH_CHECK(bias->scalar_type() == c.scalar_type() && bias->dim() == 2 && bias->size(0) == e && bias->size(1) == n &&
                    bias->is_contiguous(),
                "bias must be a contiguous [E, N] tensor of the output dtype");
  }
  const int64_t max_blocks = cdiv(sorted.numel(), block_m);
  TORCH_CHECK(experts.numel() >= max_blocks, "expert_ids is too small");
  const c10::DeviceGuard guard(a.device());
  check(sglamd_fused_moe_gemm_any(
      a.data_ptr(), a.stride(0), as.data_ptr<float>(), a_m, a_k, b.data_ptr(), b.stride(0), b.stride(1),
      bs.data_ptr<float>(), b_e, b_n, b_k, bias ? bias->data_ptr() : nullptr, n, c.data_ptr(), n, tag(c.scalar_type()),
      tag(a.scalar_type()), (int)bn, (int)bk, sorted.data_ptr<int32_t>(), experts.data_ptr<int32_t>(),
      post_pad.data_ptr<int32_t>(), topk_weights ? topk_weights->data_ptr<float>() : nullptr, num_valid, (int)top_k,
      mul_routed_weight, (int)block_m, max_blocks, n, k, stream_of(a)));
}

// One-call launcher of the whole block-FP8 MoE layer (the kernel sequence of fused_moe.py:401-785 issued from C on the
// current stream).  `workspace` is a uint8 device tensor of at least fused_moe_block_fp8_workspace_bytes(...) bytes;
// one is taken from torch's caching allocator when omitted.
void fused_moe_block_fp8_(const Tensor& hidden, const Tensor& w1, const Tensor& w2, const Tensor& w1_scale,
                          const Tensor& w2_scale, const Tensor& topk_weights, const Tensor& topk_ids, const Tensor& out,
                          double routed_scaling_factor, int64_t block_m, const optional<Tensor>& workspace) {
  const int64_t m = hidden.size(0), h = hidden.size(1), e = w1.size(0), n2 = w1.size(1), i = n2 / 2;
  const int64_t topk = topk_ids.size(1);
  TORCH_CHECK(w1.scalar_type() == kFp8 && w2.scalar_type() == kFp8, "expert weights must be Float8_e4m3fn");
  TORCH_CHECK(w1.is_contiguous() && w2.is_contiguous() && w1_scale.is_contiguous() && w2_scale.is_contiguous(),
              "expert weights and scales must be contiguous");
  TORCH_CHECK(w2.dim() == 3 && w2.size(0) == e && w2.size(1) == h && w2.size(2) == i,
              "w2 must be [E, hidden, intermediate]");
  TORCH_CHECK(w1_scale.dim() == 3 && w1_scale.size(0) == e && w1_scale.size(1) == n2 / 128 &&
                  w1_scale.size(2) == h / 128 && w2_scale.dim() == 3 && w2_scale.size(0) == e &&
                  w2_scale.size(1) == h / 128 && w2_scale.size(2) == i / 128,
              "scale shapes do not match the 128x128 blocks");
  TORCH_CHECK(w1_scale.scalar_type() == at::kFloat && w2_scale.scalar_type() == at::kFloat, "scales must be Float32");
  TORCH_CHECK(topk_weights.scalar_type() == at::kFloat && topk_weights.is_contiguous(),
              "topk_weights must be contiguous Float32");
  TORCH_CHECK((topk_ids.scalar_type() == at::kInt || topk_ids.scalar_type() == at::kLong) && topk_ids.is_contiguous(),
              "topk_ids must be contiguous int32/int64");
  TORCH_CHECK(hidden.is_contiguous() && out.is_contiguous(), "hidden_states and out must be contiguous");
  const c10::DeviceGuard guard(hidden.device());
  const int64_t need = sglamd_fused_moe_block_fp8_workspace(m, h, i, (int)e, (int)topk, (int)block_m);
  const Tensor ws = workspace ? *workspace : empty({need}, at::kByte, hidden);
  TORCH_CHECK(ws.numel() * ws.element_size() >= need, "workspace is too small");
  check(sglamd_fused_moe_block_fp8(hidden.data_ptr(), tag(hidden.scalar_type()), m, h, i, (int)e, (int)topk,
                                   w1.data_ptr(), w1_scale.data_ptr<float>(), w2.data_ptr(), w2_scale.data_ptr<float>(),
                                   topk_weights.data_ptr<float>(), topk_ids.data_ptr(), tag(topk_ids.scalar_type()),
                                   out.data_ptr(), (float)routed_scaling_factor, (int)block_m, ws.data_ptr(),
                                   ws.numel() * ws.element_size(), stream_of(hidden)));
}

// The whole MoE layer (fused_moe.py:401-785) for gated SiLU experts in one of the four weight formats: 128x128 block
// scales (block = true) or one scale per output channel, e4m3fn or int8.  block_m: 0 for the library's choice.
optional<Tensor> moe_layer(const Tensor& hidden, const Tensor& w1, const Tensor& w2, const optional<Tensor>& w1_scale,
                           const optional<Tensor>& w2_scale, const optional<Tensor>& b1, const optional<Tensor>& b2,
                           const Tensor& topk_weights, const Tensor& topk_ids, bool block, bool int8, bool inplace,
                           double routed_scaling_factor, int64_t block_m) {
  if (any_observed(hidden, w1, w2, w1_scale, w2_scale, b1, b2, topk_weights, topk_ids)) return {};
  const ScalarType t = hidden.scalar_type(), wt = int8 ? at::kChar : kFp8;
  if (hidden.dim() != 2 || !hidden.is_cuda() || !is_half(t) || !hidden.is_contiguous() || hidden.size(0) == 0) return {};
  const int64_t m = hidden.size(0), h = hidden.size(1);
  if (w1.dim() != 3 || w2.dim() != 3 || w1.scalar_type() != wt || w2.scalar_type() != wt || !w1.is_contiguous() ||
      !w2.is_contiguous() || w1.device() != hidden.device() || w2.device() != hidden.device())
    return {};
  const int64_t e = w1.size(0), n2 = w1.size(1), i = n2 / 2;
  if (w1.size(2) != h || w2.size(0) != e || w2.size(1) != h || w2.size(2) != i || h % 128 || n2 % 256 || e + 1 > 2048 ||
      h == 0 || n2 == 0)
    return {};
  auto plain_scale = [&](const optional<Tensor>& s, int64_t n, int64_t k) {
    if (!s || s->scalar_type() != at::kFloat || !s->is_contiguous() || s->device() != hidden.device()) return false;
    if (!block) return s->numel() == e * n;
    return s->dim() == 3 && s->size(0) == e && s->size(1) == n / 128 && s->size(2) == k / 128;
  };
  if (!plain_scale(w1_scale, n2, h) || !plain_scale(w2_scale, h, i)) return {};
  if (block && (b1 || b2)) return {};
  // row-scaled layers: whole rows in registers, matrices behind 32-bit buffer offsets
  if (!block && (h > 32768 || i > 32768 || n2 * h >= 0x7ffffff0ll || m * h >= 0x7ffffff0ll || m * topk_ids.size(-1) * i >= 0x7ffffff0ll))
    return {};
  auto plain_expert_bias = [&](const optional<Tensor>& b, int64_t n) {
    return !b || (b->dim() == 2 && b->size(0) == e && b->size(1) == n && b->is_contiguous() && b->scalar_type() == t &&
                  b->device() == hidden.device());
  };
  if (!plain_expert_bias(b1, n2) || !plain_expert_bias(b2, h)) return {};
  if (topk_ids.dim() != 2 || topk_ids.sizes() != topk_weights.sizes() || topk_ids.size(0) != m || topk_ids.size(1) == 0 ||
      topk_ids.device() != hidden.device() || topk_weights.device() != hidden.device() ||
      (topk_ids.scalar_type() != at::kInt && topk_ids.scalar_type() != at::kLong))
    return {};
  const int64_t topk = topk_ids.size(1);
  if (m * topk >= (1ll << 30)) return {};
  const c10::DeviceGuard guard(hidden.device());
  const Tensor tw = topk_weights.to(at::kFloat).contiguous(), ids = topk_ids.contiguous();
  Tensor out = inplace ? hidden : empty({m, h}, t, hidden);
  const int mode = block ? (int8 ? SGLAMD_MOE_BLOCK_INT8 : SGLAMD_MOE_BLOCK_FP8)
                         : (int8 ? SGLAMD_MOE_ROW_INT8 : SGLAMD_MOE_ROW_FP8);
  const int64_t need = sglamd_fused_moe_layer_workspace(mode, m, h, i, (int)e, (int)topk, (int)block_m);
  const Tensor ws = empty({need}, at::kByte, hidden);
  check(sglamd_fused_moe_layer(mode, hidden.data_ptr(), tag(t), m, h, i, (int)e, (int)topk, w1.data_ptr(),
                               w1_scale->data_ptr<float>(), b1 ? b1->data_ptr() : nullptr, w2.data_ptr(),
                               w2_scale->data_ptr<float>(), b2 ? b2->data_ptr() : nullptr, tw.data_ptr<float>(),
                               ids.data_ptr(), tag(ids.scalar_type()), out.data_ptr(), (float)routed_scaling_factor,
                               (int)block_m, ws.data_ptr(), need, stream_of(hidden)));
  if (inplace) written_in_place(hidden);
  return out;
}

// cutlass_fused_experts_fp8 (cutlass_moe.py:29-341) in its block-scaled configuration: w1 [E, k, 2n] and w2 [E, n, k] as
// column-major views of contiguous [E, 2n, k] / [E, k, n] weights, the scales as the matching views.
optional<Tensor> moe_grouped_layer(const Tensor& a, const Tensor& w1, const Tensor& w2, const Tensor& w1_scale,
                                   const Tensor& w2_scale, const Tensor& topk_weights, const Tensor& topk_ids,
                                   const Tensor& offsets, const Tensor& sizes1, const Tensor& sizes2,
                                   const optional<Tensor>& output) {
  if (any_observed(a, w1, w2, w1_scale, w2_scale, topk_weights, topk_ids, offsets, sizes1, sizes2, output)) return {};
  const ScalarType t = a.scalar_type();
  if (a.dim() != 2 || !a.is_cuda() || !is_half(t) || !a.is_contiguous() || a.size(0) == 0) return {};
  const int64_t m = a.size(0), k = a.size(1);
  // a [E, c, r] view of contiguous [E, r, c] memory
  auto column_major = [&](const Tensor& v, int64_t e, int64_t r, int64_t c, ScalarType vt) {
    return v.dim() == 3 && v.scalar_type() == vt && v.device() == a.device() && v.size(0) == e && v.size(1) == c &&
           v.size(2) == r && v.transpose(1, 2).is_contiguous();
  };
  if (w1.dim() != 3) return {};
  const int64_t e = w1.size(0), n = w1.size(2) / 2;
  if (k == 0 || n == 0 || k % 128 || n % 128 || w1.size(2) % 2 || e + 1 > 2048) return {};
  if (!column_major(w1, e, 2 * n, k, kFp8) || !column_major(w2, e, k, n, kFp8) ||
      !column_major(w1_scale, e, 2 * n / 128, k / 128, at::kFloat) ||
      !column_major(w2_scale, e, k / 128, n / 128, at::kFloat))
    return {};
  if (topk_ids.dim() != 2 || topk_ids.scalar_type() != at::kInt || !topk_ids.is_contiguous() || topk_ids.size(0) != m ||
      topk_ids.size(1) == 0 || topk_ids.sizes() != topk_weights.sizes() || topk_ids.device() != a.device() ||
      topk_weights.device() != a.device() || m * topk_ids.size(1) >= (1ll << 30))
    return {};
  auto table = [&](const Tensor& v, int64_t need) {
    return v.scalar_type() == at::kInt && v.is_contiguous() && v.numel() >= need && v.device() == a.device();
  };
  if (!table(offsets, e + 1) || !table(sizes1, 3 * e) || !table(sizes2, 3 * e)) return {};
  if (output && !(output->sizes() == a.sizes() && output->scalar_type() == t && output->is_contiguous() &&
                  output->device() == a.device()))
    return {};
  const int64_t topk = topk_ids.size(1);
  const c10::DeviceGuard guard(a.device());
  const Tensor tw = topk_weights.to(at::kFloat).contiguous();
  Tensor out = output ? *output : empty({m, k}, t, a);
  const int64_t need = sglamd_fused_moe_layer_workspace(SGLAMD_MOE_BLOCK_FP8, m, k, n, (int)e, (int)topk, 0);
  const Tensor ws = empty({need}, at::kByte, a);
  check(sglamd_fused_moe_grouped_layer(a.data_ptr(), tag(t), m, k, n, (int)e, (int)topk, w1.data_ptr(),
                                       w1_scale.data_ptr<float>(), w2.data_ptr(), w2_scale.data_ptr<float>(),
                                       tw.data_ptr<float>(), topk_ids.data_ptr<int32_t>(), offsets.data_ptr<int32_t>(),
                                       sizes1.data_ptr<int32_t>(), sizes2.data_ptr<int32_t>(), out.data_ptr(),
                                       ws.data_ptr(), need, stream_of(a)));
  return out;
}

}  // namespace

TORCH_LIBRARY_FRAGMENT(sgl_kernel, m) {
  m.def(
      "sgl_per_token_group_quant_8bit(Tensor input, Tensor! output_q, Tensor! output_s, int group_size, float eps, "
      "float fp8_min, float fp8_max, bool scale_ue8m0) -> ()");
  m.def(
      "sgl_per_token_group_quant_8bit_v2(Tensor input, Tensor! output_q, Tensor! output_s, int group_size, float eps, "
      "float fp8_min, float fp8_max, bool scale_ue8m0, bool fuse_silu_and_mul, Tensor? masked_m) -> ()");
  m.def("sgl_per_token_quant_fp8(Tensor input, Tensor! output_q, Tensor! output_s) -> ()");
  m.def(
      "fp8_blockwise_scaled_mm(Tensor mat_a, Tensor mat_b, Tensor scales_a, Tensor scales_b, ScalarType out_dtype) -> "
      "Tensor");
  m.def(
      "fp8_scaled_mm(Tensor mat_a, Tensor mat_b, Tensor scales_a, Tensor scales_b, ScalarType out_dtype, Tensor? bias) "
      "-> Tensor");
  m.def(
      "int8_scaled_mm(Tensor mat_a, Tensor mat_b, Tensor scales_a, Tensor scales_b, ScalarType out_dtype, Tensor? "
      "bias) -> Tensor");
  m.def(
      "topk_softmax(Tensor! topk_weights, Tensor! topk_indices, Tensor gating_output, bool renormalize, float "
      "moe_softcapping, Tensor? correction_bias) -> ()");
  m.def(
      "topk_sigmoid(Tensor! topk_weights, Tensor! topk_indices, Tensor gating_output, bool renormalize, Tensor? "
      "correction_bias) -> ()");
  m.def(
      "moe_align_block_size(Tensor topk_ids, int num_experts, int block_size, Tensor! sorted_token_ids, Tensor! "
      "experts_ids, Tensor! num_tokens_post_pad, Tensor! cumsum_buffer, bool pad_sorted_token_ids) -> ()");
  m.def("silu_and_mul(Tensor! out, Tensor input) -> ()");
  m.def("gelu_tanh_and_mul(Tensor! out, Tensor input) -> ()");
  m.def("gelu_and_mul(Tensor! out, Tensor input) -> ()");
  m.def("moe_sum_reduce(Tensor input, Tensor output, float routed_scaling_factor) -> ()");
  m.def(
      "prepare_moe_input(Tensor topk_ids, Tensor expert_offsets, Tensor? blockscale_offsets, Tensor problem_sizes1, "
      "Tensor problem_sizes2, Tensor input_permutation, Tensor output_permutation, int num_experts, int n, int k) -> "
      "()");
  m.def("shuffle_rows(Tensor input, Tensor dst2src_map, Tensor output) -> ()");
  m.def("apply_shuffle_mul_sum(Tensor input, Tensor output, Tensor permutation, Tensor? factors) -> ()");
  m.def(
      "fp8_blockwise_scaled_grouped_mm(Tensor output, Tensor a_ptrs, Tensor b_ptrs, Tensor out_ptrs, Tensor "
      "a_scales_ptrs, Tensor b_scales_ptrs, Tensor a, Tensor b, Tensor scales_a, Tensor scales_b, Tensor stride_a, "
      "Tensor stride_b, Tensor stride_c, Tensor layout_sfa, Tensor layout_sfb, Tensor problem_sizes, Tensor "
      "expert_offsets, Tensor workspace) -> ()");
  m.def(
      "es_fp8_blockwise_scaled_grouped_mm(Tensor output, Tensor a, Tensor b, Tensor scales_a, Tensor scales_b, Tensor "
      "stride_a, Tensor stride_b, Tensor stride_d, Tensor problem_sizes, Tensor expert_offsets, Tensor workspace) -> "
      "()");
}

TORCH_LIBRARY_IMPL(sgl_kernel, CUDA, m) {
  m.impl("sgl_per_token_group_quant_8bit", sgl_per_token_group_quant_8bit);
  m.impl("sgl_per_token_group_quant_8bit_v2", sgl_per_token_group_quant_8bit_v2);
  m.impl("sgl_per_token_quant_fp8", sgl_per_token_quant_fp8);
  m.impl("fp8_blockwise_scaled_mm", fp8_blockwise_scaled_mm);
  m.impl("fp8_scaled_mm", fp8_scaled_mm);
  m.impl("int8_scaled_mm", int8_scaled_mm);
  m.impl("topk_softmax", topk_softmax);
  m.impl("topk_sigmoid", topk_sigmoid);
  m.impl("moe_align_block_size", moe_align_block_size);
  m.impl("silu_and_mul", silu_and_mul);
  m.impl("gelu_tanh_and_mul", gelu_tanh_and_mul);
  m.impl("gelu_and_mul", gelu_and_mul);
  m.impl("moe_sum_reduce", moe_sum_reduce);
  m.impl("prepare_moe_input", prepare_moe_input);
  m.impl("shuffle_rows", shuffle_rows);
  m.impl("apply_shuffle_mul_sum", apply_shuffle_mul_sum);
  m.impl("fp8_blockwise_scaled_grouped_mm", fp8_blockwise_scaled_grouped_mm);
  m.impl("es_fp8_blockwise_scaled_grouped_mm", es_fp8_blockwise_scaled_grouped_mm);
}

// A launch may wait for room in the stream's queue: other Python threads run meanwhile.
using Unlocked = py::call_guard<py::gil_scoped_release>;

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("set_error_type", [](py::object type) { g_error_type = type.release().ptr(); });
  m.def("static_quant_fp8_", &static_quant_fp8_, Unlocked(), py::arg("input"), py::arg("output_q"), py::arg("scale"),
        py::arg("scale_rows") = py::none());
  m.def("tensor_absmax_scale_", &tensor_absmax_scale_, Unlocked(), py::arg("input"), py::arg("scale"), py::arg("eps") = 1e-12,
        py::arg("fp8_max") = 448.0);
  m.def("per_token_quant_int8_", &per_token_quant_int8_, Unlocked());
  m.def("ue8m0_unpack_", &ue8m0_unpack_, Unlocked(), py::arg("packed"), py::arg("rows"), py::arg("groups"), py::arg("row_step") = 1);
  m.def("any_observed", [](const std::vector<optional<Tensor>>& tensors) {
    return is_observed() || std::any_of(tensors.begin(), tensors.end(), [](const auto& t) { return is_observed(t); });
  });
  m.def("written_in_place", &written_in_place);
  m.def("group_quant_2d", &group_quant_2d, Unlocked());
  m.def("per_token_quant", &per_token_quant, Unlocked());
  m.def("fused_rms_group_quant", &fused_rms_group_quant, Unlocked());
  m.def("w8a8_block_fp8_matmul_", &w8a8_block_fp8_matmul_, Unlocked(), py::arg("A"), py::arg("B"), py::arg("As"), py::arg("Bs"),
        py::arg("C"), py::arg("pow2_scales") = false);
  m.def("w8a8_block_int8_matmul_", &w8a8_block_int8_matmul_, Unlocked());
  m.def("block_scaled_mm_any_", &block_scaled_mm_any_, Unlocked());
  m.def("block_linear", &block_linear, Unlocked());
  m.def("block_matmul", &block_matmul, Unlocked());
  m.def("row_linear", &row_linear, Unlocked());
  m.def("fused_moe_block_fp8_gemm_", &fused_moe_block_fp8_gemm_, Unlocked());
  m.def("fused_moe_gemm_any_", &fused_moe_gemm_any_, Unlocked(), py::arg("A"), py::arg("A_scale"), py::arg("B"), py::arg("B_scale"),
        py::arg("C"), py::arg("topk_weights"), py::arg("sorted_token_ids"), py::arg("expert_ids"),
        py::arg("num_tokens_post_padded"), py::arg("mul_routed_weight"), py::arg("top_k"), py::arg("block_m"),
        py::arg("block_shape") = py::none(), py::arg("bias") = py::none());
  m.def("fused_moe_block_fp8_", &fused_moe_block_fp8_, Unlocked(), py::arg("hidden_states"), py::arg("w1"), py::arg("w2"),
        py::arg("w1_scale"), py::arg("w2_scale"), py::arg("topk_weights"), py::arg("topk_ids"), py::arg("out"),
        py::arg("routed_scaling_factor"), py::arg("block_m") = 0, py::arg("workspace") = py::none());
  m.def("moe_layer", &moe_layer, Unlocked());
  m.def("moe_grouped_layer", &moe_grouped_layer, Unlocked());
  m.def("fused_moe_block_fp8_workspace_bytes",
        [](int64_t m_, int64_t h, int64_t i, int64_t e, int64_t topk, int64_t block_m) {
          return sglamd_fused_moe_block_fp8_workspace(m_, h, i, (int)e, (int)topk, (int)block_m);
        },
        py::arg("M"), py::arg("H"), py::arg("I"), py::arg("E"), py::arg("topk"), py::arg("block_m") = 0);
}
