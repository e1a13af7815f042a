// GPU kernels of the mpk:: torch operators: output allocation, alignment checks and the C ABI
// call (include/mpk.h) on torch's current stream.
//
// The operators themselves (schemas, fake kernels, autograd behaviour) are defined in Python
// (_ops.py, torch.library.custom_op); this library registers their CUDA-key kernels, which the
// dispatcher reaches below autograd, tracing and functorch as it did the Python bodies before.
// What it saves is host time: a Python body cost 8-30 us of interpreter, ctypes and tensor
// wrapper work per launch, more than most launches of a small forward take on the GPU.
// Measured on MI355X in inference mode, us per call among others, before -> after:
// 77 x 2048 x 512 projection + GELU 15.9 -> 7.8, layer tail over 4099 x 64 36.8 -> 15.7, forward of
// B1 S128 D128 L4 (9 launches) 277 -> 112 (with each module attribute looked up once in the wrappers).
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/library.h>

#include <optional>
#include <tuple>

#include "mpk.h"

namespace {

using at::Tensor;

void check(int status, const char* what) {
  TORCH_CHECK(status == MPK_OK, what, " failed with status ", status, ": ", mpk_status_string(status));
}

at::ScalarType scalar_type(int64_t code) {
  TORCH_CHECK_VALUE(code == MPK_F32 || code == MPK_F16, "unknown dtype code ", code);
  return code == MPK_F16 ? at::kHalf : at::kFloat;
}

int dtype_code(const Tensor& t) {
  TORCH_CHECK_VALUE(t.scalar_type() == at::kHalf || t.scalar_type() == at::kFloat, "unsupported dtype ",
                    t.scalar_type());
  return t.scalar_type() == at::kHalf ? MPK_F16 : MPK_F32;
}

template <typename... T>
void require_aligned(const char* message, const T&... tensors) {
  const uintptr_t bits = (reinterpret_cast<uintptr_t>(tensors.data_ptr()) | ... | uintptr_t{0});
  TORCH_CHECK_VALUE(bits % 16 == 0, message, " (16-byte alignment)");
}

const void* ptr(const std::optional<Tensor>& t) { return t.has_value() ? t->data_ptr() : nullptr; }
const float* f32(const Tensor& t) { return static_cast<const float*>(t.data_ptr()); }
float* f32_out(const Tensor& t) { return static_cast<float*>(t.data_ptr()); }
void* stream(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
int64_t rows(const Tensor& t, int64_t width) { return width ? t.numel() / width : 0; }

// a contiguous output of t's shape with the last dimension replaced by `width`
Tensor empty_rows(const Tensor& t, int64_t width, at::ScalarType dtype) {
  c10::DimVector sizes(t.sizes().begin(), t.sizes().end());
  if (sizes.empty()) sizes.resize(1);  // a 0-d tensor has rows of width 1
  sizes.back() = width;
  return at::empty(sizes, t.options().dtype(dtype));
}

Tensor layer_norm(const Tensor& x, const Tensor& weight, const Tensor& bias, double eps, int64_t out_dtype) {
  const c10::DeviceGuard guard(x.device());
  const int64_t d = x.size(-1);
  Tensor out = empty_rows(x, d, scalar_type(out_dtype));
  require_aligned("unsupported LayerNorm inputs", x, weight, bias, out);
  check(mpk_layernorm(f32(x), nullptr, f32(weight), f32(bias), nullptr, out.data_ptr(), (int)out_dtype, rows(x, d),
                      (int32_t)d, (float)eps, stream(x)),
        "mpk_layernorm");
  return out;
}

std::tuple<Tensor, Tensor> add_layer_norm(const Tensor& x, const Tensor& update, const Tensor& weight,
                                          const Tensor& bias, double eps, int64_t out_dtype) {
  const c10::DeviceGuard guard(x.device());
  const int64_t d = x.size(-1);
  Tensor residual = at::empty_like(x);
  Tensor out = empty_rows(x, d, scalar_type(out_dtype));
  require_aligned("unsupported residual/LayerNorm inputs", x, update, weight, bias, residual, out);
  check(mpk_layernorm(f32(x), f32(update), f32(weight), f32(bias), f32_out(residual), out.data_ptr(), (int)out_dtype,
                      rows(x, d), (int32_t)d, (float)eps, stream(x)),
        "mpk_layernorm");
  return {residual, out};
}

Tensor linear(const Tensor& x, const Tensor& weight, const Tensor& bias, int64_t out_dtype, bool gelu,
              int64_t variant) {
  const c10::DeviceGuard guard(x.device());
  const int64_t n = weight.size(0), k = weight.size(1);
  Tensor out = empty_rows(x, n, scalar_type(out_dtype));
  require_aligned("unsupported mixed projection inputs", x, weight, bias, out);
  check(mpk_linear(x.data_ptr(), dtype_code(x), weight.data_ptr(), bias.data_ptr(), out.data_ptr(), (int)out_dtype,
                   gelu ? 1 : 0, rows(x, k), (int32_t)n, (int32_t)k, (int)variant, stream(x)),
        "mpk_linear");
  return out;
}

Tensor linear_qscaled(const Tensor& x, const Tensor& weight, const Tensor& bias, int64_t out_dtype, int64_t q_cols,
                      double q_scale, int64_t variant) {
  const c10::DeviceGuard guard(x.device());
  const int64_t n = weight.size(0), k = weight.size(1);
  Tensor out = empty_rows(x, n, scalar_type(out_dtype));
  require_aligned("unsupported mixed projection inputs", x, weight, bias, out);
  check(mpk_linear_qscaled(x.data_ptr(), dtype_code(x), weight.data_ptr(), bias.data_ptr(), out.data_ptr(),
                           (int)out_dtype, rows(x, k), (int32_t)n, (int32_t)k, (int32_t)q_cols, (float)q_scale,
                           (int)variant, stream(x)),
        "mpk_linear_qscaled");
  return out;
}

void linear_residual_into(const Tensor& x, const Tensor& weight, const Tensor& bias, const Tensor& residual,
                          const Tensor& out, int64_t variant) {
  const c10::DeviceGuard guard(x.device());
  const int64_t n = weight.size(0), k = weight.size(1);
  require_aligned("unsupported mixed projection/residual inputs", x, weight, bias, residual, out);
  check(mpk_linear_residual(x.data_ptr(), dtype_code(x), weight.data_ptr(), bias.data_ptr(), f32(residual),
                            f32_out(out), rows(x, k), (int32_t)n, (int32_t)k, (int)variant, stream(x)),
        "mpk_linear_residual");
}

Tensor linear_residual(const Tensor& x, const Tensor& weight, const Tensor& bias, const Tensor& residual,
                       int64_t variant) {
  Tensor out = at::empty_like(residual);
  linear_residual_into(x, weight, bias, residual, out, variant);
  return out;
}

std::tuple<Tensor, Tensor> linear_residual_layer_norm(const Tensor& x, const Tensor& weight, const Tensor& bias,
                                                      const Tensor& residual, const Tensor& gamma, const Tensor& beta,
                                                      double eps, int64_t out_dtype, int64_t variant) {
  const c10::DeviceGuard guard(x.device());
  const int64_t d = weight.size(0);
  Tensor residual_out = at::empty_like(residual);
  Tensor normalized = empty_rows(residual, residual.size(-1), scalar_type(out_dtype));
  require_aligned("unsupported fused projection/residual/LayerNorm inputs", x, weight, bias, residual, gamma, beta,
                  residual_out, normalized);
  check(mpk_linear_residual_layernorm(x.data_ptr(), dtype_code(x), weight.data_ptr(), bias.data_ptr(), f32(residual),
                                      f32(gamma), f32(beta), f32_out(residual_out), normalized.data_ptr(),
                                      (int)out_dtype, rows(x, d), (int32_t)d, (float)eps, (int)variant, stream(x)),
        "mpk_linear_residual_layernorm");
  return {residual_out, normalized};
}

std::tuple<Tensor, Tensor> linear_add_layer_norm(const Tensor& x, const Tensor& weight, const Tensor& bias,
                                                 const Tensor& residual, const Tensor& gamma, const Tensor& beta,
                                                 double eps, int64_t out_dtype) {
  const c10::DeviceGuard guard(x.device());
  const int64_t n = weight.size(0), k = weight.size(1);
  Tensor residual_out = at::empty_like(residual);
  Tensor normalized = empty_rows(residual, residual.size(-1), scalar_type(out_dtype));
  require_aligned("unsupported projection/residual/LayerNorm inputs", x, weight, bias, residual, gamma, beta,
                  residual_out, normalized);
  check(mpk_linear_add_layernorm(x.data_ptr(), dtype_code(x), weight.data_ptr(), bias.data_ptr(), f32(residual),
                                 f32(gamma), f32(beta), f32_out(residual_out), normalized.data_ptr(), (int)out_dtype,
                                 rows(residual, n), (int32_t)n, (int32_t)k, (float)eps, stream(x)),
        "mpk_linear_add_layernorm");
  return {residual_out, normalized};
}

// FP16 FFNs at d_model 256 / 512 up to these row counts run as projection + GELU (hidden in a
// temporary of at most 512 MB from torch's caching allocator), projection + residual, and
// LayerNorm.  The fused kernels walk the hidden layer in 32-wide chunks on one workgroup per
// 128 tokens (d 256) or 64 (d 512), so a short call takes as long as a full device of rows.
// Measured on MI355X, us, fused -> separate: d 256, F 1024: 16 rows
// 42.8 -> 11.9, 4,096 50.9 -> 19.8, 16,384 52.6 -> 44.3, 32,768 59.6 -> 74.7; F 256: 4,096
// 24.6 -> 13.6, 16,384 26.7 -> 24.4, 32,768 29.6 -> 42.6; d 512, F 2048: slower fused at every
// row count (32,768: 848 -> 214).
constexpr int64_t kSplitFfnRows256 = 16384;
constexpr int64_t kSplitFfnHidden = int64_t{1} << 28;  // elements

bool split_ffn(const Tensor& x, int64_t d, int64_t f, int64_t variant) {
  return variant == 0 && x.scalar_type() == at::kHalf && f % 64 == 0 &&
         rows(x, d) * f <= kSplitFfnHidden && (d == 512 || (d == 256 && rows(x, d) <= kSplitFfnRows256));
}

// residual_out undefined: only `normalized` is stored
void launch_ffn(const Tensor& x, const Tensor& w_in, const Tensor& b_in, const Tensor& w_out, const Tensor& b_out,
                const Tensor& residual, const Tensor& gamma, const Tensor& beta, double eps, int64_t variant,
                const Tensor& residual_out, const Tensor& normalized) {
  const int64_t f = w_in.size(0), d = w_in.size(1);
  require_aligned("unsupported fused FFN inputs", x, w_in, b_in, w_out, b_out, residual, gamma, beta, normalized);
  if (residual_out.defined()) require_aligned("unsupported fused FFN inputs", residual_out);
  if (split_ffn(x, d, f, variant)) {
    const int64_t m = rows(x, d);
    const Tensor hidden = at::empty({m, f}, x.options());
    const Tensor r = residual_out.defined() ? residual_out : at::empty_like(residual);
    check(mpk_linear(x.data_ptr(), MPK_F16, w_in.data_ptr(), b_in.data_ptr(), hidden.data_ptr(), MPK_F16, 1, m,
                     (int32_t)f, (int32_t)d, 0, stream(x)),
          "mpk_linear");
    check(mpk_linear_residual(hidden.data_ptr(), MPK_F16, w_out.data_ptr(), b_out.data_ptr(), f32(residual),
                              f32_out(r), m, (int32_t)d, (int32_t)f, 0, stream(x)),
          "mpk_linear_residual");
    check(mpk_layernorm(f32(r), nullptr, f32(gamma), f32(beta), nullptr, normalized.data_ptr(),
                        dtype_code(normalized), m, (int32_t)d, (float)eps, stream(x)),
          "mpk_layernorm");
    return;
  }
  check(mpk_ffn_residual_layernorm(x.data_ptr(), dtype_code(x), w_in.data_ptr(), b_in.data_ptr(), w_out.data_ptr(),
                                   b_out.data_ptr(), f32(residual), f32(gamma), f32(beta),
                                   residual_out.defined() ? f32_out(residual_out) : nullptr, normalized.data_ptr(),
                                   dtype_code(normalized), rows(x, d), (int32_t)d, (int32_t)f, (float)eps,
                                   (int)variant, stream(x)),
        "mpk_ffn_residual_layernorm");
}

std::tuple<Tensor, Tensor> ffn_residual_layer_norm(const Tensor& x, const Tensor& w_in, const Tensor& b_in,
                                                   const Tensor& w_out, const Tensor& b_out, const Tensor& residual,
                                                   const Tensor& gamma, const Tensor& beta, double eps,
                                                   int64_t out_dtype, int64_t variant) {
  const c10::DeviceGuard guard(x.device());
  Tensor residual_out = at::empty_like(residual);
  Tensor normalized = empty_rows(residual, residual.size(-1), scalar_type(out_dtype));
  launch_ffn(x, w_in, b_in, w_out, b_out, residual, gamma, beta, eps, variant, residual_out, normalized);
  return {residual_out, normalized};
}

Tensor ffn_residual_layer_norm_into(const Tensor& x, const Tensor& w_in, const Tensor& b_in, const Tensor& w_out,
                                    const Tensor& b_out, const Tensor& residual, const Tensor& gamma,
                                    const Tensor& beta, double eps, int64_t variant, const Tensor& normalized,
                                    bool store_residual) {
  const c10::DeviceGuard guard(x.device());
  Tensor residual_out = store_residual ? at::empty_like(residual) : Tensor();
  launch_ffn(x, w_in, b_in, w_out, b_out, residual, gamma, beta, eps, variant, residual_out, normalized);
  return store_residual ? residual_out : at::empty({0}, residual.options());
}

Tensor ffn_residual_layer_norm_final(const Tensor& x, const Tensor& w_in, const Tensor& b_in, const Tensor& w_out,
                                     const Tensor& b_out, const Tensor& residual, const Tensor& gamma,
                                     const Tensor& beta, double eps, int64_t out_dtype, int64_t variant) {
  const c10::DeviceGuard guard(x.device());
  Tensor normalized = empty_rows(residual, residual.size(-1), scalar_type(out_dtype));
  launch_ffn(x, w_in, b_in, w_out, b_out, residual, gamma, beta, eps, variant, Tensor(), normalized);
  return normalized;
}

// contiguous [B, S, H, hd] output of [B, H, S, hd] views, and its strides in their order
Tensor attention_out(const Tensor& q, at::ScalarType dtype, int64_t (&strides)[4]) {
  const int64_t b = q.size(0), h = q.size(1), s = q.size(2), hd = q.size(3);
  strides[0] = s * h * hd, strides[1] = hd, strides[2] = h * hd, strides[3] = 1;
  return at::empty({b, s, h, hd}, q.options().dtype(dtype));
}

void require_aligned_qkv(const Tensor& q, const Tensor& k, const Tensor& v) {
  TORCH_CHECK_VALUE(q.dim() == 4 && k.dim() == 4 && v.dim() == 4, "unsupported custom-attention input: shape=",
                    q.sizes(), ", dtype=", q.scalar_type(), " (4 dimensions)");
  const uintptr_t bits = reinterpret_cast<uintptr_t>(q.data_ptr()) | reinterpret_cast<uintptr_t>(k.data_ptr()) |
                         reinterpret_cast<uintptr_t>(v.data_ptr());
  TORCH_CHECK_VALUE(bits % 16 == 0, "unsupported custom-attention input: shape=", q.sizes(), ", dtype=",
                    q.scalar_type(), " (16-byte alignment)");
}

Tensor attention(const Tensor& q, const Tensor& k, const Tensor& v, const std::optional<Tensor>& key_valid,
                 double scale, bool causal, int64_t out_dtype, int64_t variant) {
  const c10::DeviceGuard guard(q.device());
  require_aligned_qkv(q, k, v);
  int64_t os[4];
  Tensor out = attention_out(q, scalar_type(out_dtype), os);
  check(mpk_causal_attention(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), dtype_code(q), (int)out_dtype,
                             q.strides().data(), k.strides().data(), v.strides().data(), os, (int32_t)q.size(0),
                             (int32_t)q.size(1), (int32_t)q.size(2), (int32_t)q.size(3), (float)scale, causal ? 1 : 0,
                             static_cast<const uint8_t*>(ptr(key_valid)), (int)variant, stream(q)),
        "mpk_causal_attention");
  return out;
}

Tensor attention_prescaled(const Tensor& q, const Tensor& k, const Tensor& v, const std::optional<Tensor>& key_valid,
                           bool causal, int64_t out_dtype, int64_t variant) {
  const c10::DeviceGuard guard(q.device());
  require_aligned_qkv(q, k, v);
  int64_t os[4];
  Tensor out = attention_out(q, scalar_type(out_dtype), os);
  check(mpk_causal_attention_prescaled(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), (int)out_dtype,
                                       q.strides().data(), k.strides().data(), v.strides().data(), os,
                                       (int32_t)q.size(0), (int32_t)q.size(1), (int32_t)q.size(2),
                                       (int32_t)q.size(3), causal ? 1 : 0,
                                       static_cast<const uint8_t*>(ptr(key_valid)), (int)variant, stream(q)),
        "mpk_causal_attention_prescaled");
  return out;
}

Tensor layer_norm_qkv(const Tensor& x, const Tensor& ln_w, const Tensor& ln_b, const Tensor& w_qkv,
                      const Tensor& b_qkv, double eps, int64_t variant, double q_scale) {
  const c10::DeviceGuard guard(x.device());
  const int64_t d = x.size(-1);
  Tensor out = empty_rows(x, 3 * d, at::kHalf);
  require_aligned("unsupported LayerNorm/QKV inputs", x, ln_w, ln_b, w_qkv, b_qkv, out);
  if (q_scale != 0.0)
    check(mpk_layernorm_qkv_qscaled(f32(x), f32(ln_w), f32(ln_b), w_qkv.data_ptr(), b_qkv.data_ptr(), out.data_ptr(),
                                    rows(x, d), (int32_t)d, (float)eps, (float)q_scale, (int)variant, stream(x)),
          "mpk_layernorm_qkv_qscaled");
  else
    check(mpk_layernorm_qkv(f32(x), f32(ln_w), f32(ln_b), w_qkv.data_ptr(), b_qkv.data_ptr(), out.data_ptr(),
                            rows(x, d), (int32_t)d, (float)eps, (int)variant, stream(x)),
          "mpk_layernorm_qkv");
  return out;
}

// the layer-tail operators' tensor list
struct TailTensors {
  const Tensor &w_o, &b_o, &ln2_w, &ln2_b, &w_in, &b_in, &w_out, &b_out, &next_w, &next_b;
  explicit TailTensors(at::TensorList t)
      : w_o(at10(t)[0]), b_o(t[1]), ln2_w(t[2]), ln2_b(t[3]), w_in(t[4]), b_in(t[5]), w_out(t[6]), b_out(t[7]),
        next_w(t[8]), next_b(t[9]) {}
  static at::TensorList at10(at::TensorList t) {
    TORCH_CHECK_VALUE(t.size() == 10, "expected 10 layer-tail tensors, got ", t.size());
    return t;
  }
};

void require_aligned_tail(const char* message, at::TensorList tensors, const std::optional<Tensor>& w_qkv,
                          const std::optional<Tensor>& b_qkv) {
  uintptr_t bits = reinterpret_cast<uintptr_t>(ptr(w_qkv)) | reinterpret_cast<uintptr_t>(ptr(b_qkv));
  for (const Tensor& t : tensors) bits |= reinterpret_cast<uintptr_t>(t.data_ptr());
  TORCH_CHECK_VALUE(bits % 16 == 0, message, " (16-byte alignment)");
}

std::tuple<Tensor, Tensor> layer_tail(const Tensor& ctx, const Tensor& residual, at::TensorList tensors,
                                      const std::optional<Tensor>& w_qkv, const std::optional<Tensor>& b_qkv,
                                      double ln2_eps, double next_eps, int64_t variant, double q_scale) {
  const c10::DeviceGuard guard(ctx.device());
  const TailTensors t(tensors);
  const int64_t d = ctx.size(-1), f = t.w_in.size(0);
  const bool last = !w_qkv.has_value();
  Tensor residual_out = at::empty_like(residual);
  Tensor out = empty_rows(ctx, last ? d : 3 * d, last ? at::kFloat : at::kHalf);
  const char* message = "unsupported fused layer-tail inputs";
  require_aligned(message, ctx, residual, residual_out, out);
  require_aligned_tail(message, tensors, w_qkv, b_qkv);
  if (q_scale != 0.0)
    check(mpk_layer_tail_qscaled(ctx.data_ptr(), f32(residual), t.w_o.data_ptr(), t.b_o.data_ptr(), f32(t.ln2_w),
                                 f32(t.ln2_b), t.w_in.data_ptr(), t.b_in.data_ptr(), t.w_out.data_ptr(),
                                 t.b_out.data_ptr(), f32(t.next_w), f32(t.next_b), ptr(w_qkv), ptr(b_qkv),
                                 f32_out(residual_out), out.data_ptr(), last ? 1 : 0, rows(ctx, d), (int32_t)d,
                                 (int32_t)f, (float)ln2_eps, (float)next_eps, (float)q_scale, (int)variant,
                                 stream(ctx)),
          "mpk_layer_tail_qscaled");
  else
    check(mpk_layer_tail(ctx.data_ptr(), f32(residual), t.w_o.data_ptr(), t.b_o.data_ptr(), f32(t.ln2_w),
                         f32(t.ln2_b), t.w_in.data_ptr(), t.b_in.data_ptr(), t.w_out.data_ptr(), t.b_out.data_ptr(),
                         f32(t.next_w), f32(t.next_b), ptr(w_qkv), ptr(b_qkv), f32_out(residual_out), out.data_ptr(),
                         last ? 1 : 0, rows(ctx, d), (int32_t)d, (int32_t)f, (float)ln2_eps, (float)next_eps,
                         (int)variant, stream(ctx)),
          "mpk_layer_tail");
  return {residual_out, out};
}

std::tuple<Tensor, Tensor> attention_layer_tail(const Tensor& qkv, const Tensor& residual, at::TensorList tensors,
                                                const std::optional<Tensor>& w_qkv,
                                                const std::optional<Tensor>& b_qkv, int64_t heads, double scale,
                                                bool causal, double ln2_eps, double next_eps) {
  const c10::DeviceGuard guard(qkv.device());
  const TailTensors t(tensors);
  const int64_t d = residual.size(-1), f = t.w_in.size(0);
  const bool last = !w_qkv.has_value();
  Tensor residual_out = at::empty_like(residual);
  Tensor out = empty_rows(residual, last ? d : 3 * d, last ? at::kFloat : at::kHalf);
  const char* message = "unsupported fused attention layer-tail inputs";
  require_aligned(message, qkv, residual, residual_out, out);
  require_aligned_tail(message, tensors, w_qkv, b_qkv);
  check(mpk_attention_layer_tail(qkv.data_ptr(), f32(residual), t.w_o.data_ptr(), t.b_o.data_ptr(), f32(t.ln2_w),
                                 f32(t.ln2_b), t.w_in.data_ptr(), t.b_in.data_ptr(), t.w_out.data_ptr(),
                                 t.b_out.data_ptr(), f32(t.next_w), f32(t.next_b), ptr(w_qkv), ptr(b_qkv),
                                 f32_out(residual_out), out.data_ptr(), last ? 1 : 0, rows(residual, d), (int32_t)d,
                                 (int32_t)f, (int32_t)heads, (int32_t)residual.size(-2), (float)scale, causal ? 1 : 0,
                                 (float)ln2_eps, (float)next_eps, stream(qkv)),
        "mpk_attention_layer_tail");
  return {residual_out, out};
}

}  // namespace

TORCH_LIBRARY_IMPL(mpk, CUDA, m) {
  m.impl("layer_norm", layer_norm);
  m.impl("add_layer_norm", add_layer_norm);
  m.impl("linear", linear);
  m.impl("linear_qscaled", linear_qscaled);
  m.impl("linear_residual", linear_residual);
  m.impl("linear_residual_into", linear_residual_into);
  m.impl("linear_residual_layer_norm", linear_residual_layer_norm);
  m.impl("linear_add_layer_norm", linear_add_layer_norm);
  m.impl("ffn_residual_layer_norm", ffn_residual_layer_norm);
  m.impl("ffn_residual_layer_norm_into", ffn_residual_layer_norm_into);
  m.impl("ffn_residual_layer_norm_final", ffn_residual_layer_norm_final);
  m.impl("attention", attention);
  m.impl("attention_prescaled", attention_prescaled);
  m.impl("layer_norm_qkv", layer_norm_qkv);
  m.impl("layer_tail", layer_tail);
  m.impl("attention_layer_tail", attention_layer_tail);
}
