// Device implementations of the torch.ops.joyomni_ops operators: argument checks worded like the
// reference's TORCH_CHECKs (joyomni_ops/csrc/joyomni_ops.h:8-15 and the checks of each op's entry,
// cited below), output and workspace allocation from torch's caching allocator, then one call into
// the C ABI (include/joyomni_hip.h) on the caller's current stream. The schemas and the FakeTensor
// kernels are in joyomni_ops/__init__.py. Stateless: nothing is kept between calls.
//
// Host code in C++ because the calls of the condition stream and of small chunks are bound by it: a
// call through a Python implementation (dispatch, checks, ctypes) took 11 us for the quantiser, 18 for
// the GEMM, 21 for attention and 35 for the fused QKV projection, longer than their kernels; here 4.4,
// 7.0, 5.3 and 11.5 us (Fp8Linear on 64 rows 38.1 -> 17.9 us a call).
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/library.h>

#include <algorithm>
#include <cmath>
#include <string>
#include <tuple>

#include "../../include/joyomni_hip.h"

namespace {

using at::ScalarType;
using at::Tensor;
using OptTensor = std::optional<Tensor>;

std::string dtype_name(ScalarType t) {  // as Python prints a torch.dtype
  switch (t) {
    case at::kBFloat16: return "torch.bfloat16";
    case at::kHalf: return "torch.float16";
    case at::kFloat: return "torch.float32";
    case at::kDouble: return "torch.float64";
    case at::kFloat8_e4m3fn: return "torch.float8_e4m3fn";
    case at::kByte: return "torch.uint8";
    case at::kChar: return "torch.int8";
    case at::kShort: return "torch.int16";
    case at::kInt: return "torch.int32";
    case at::kLong: return "torch.int64";
    case at::kBool: return "torch.bool";
    default: return std::string("torch.") + c10::toString(t);
  }
}

void check_input(const Tensor& t, const char* name, ScalarType dtype) {
  TORCH_CHECK(t.is_cuda(), name, " must be a CUDA tensor");
  TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
  TORCH_CHECK(t.scalar_type() == dtype, name, " dtype is ", dtype_name(t.scalar_type()), ", expected ",
              dtype_name(dtype));
}

void* stream_of(const Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.get_device()).stream(); }
void* ptr(const Tensor& t) { return t.data_ptr(); }
void* ptr(const OptTensor& t) { return t ? t->data_ptr() : nullptr; }

// A C-ABI refusal is the package's JoyError (a RuntimeError; the argument checks here raise RuntimeError
// itself). The caller may have released the GIL.
void check_status(joy_status st) {
  if (st == JOY_OK) return;
  const PyGILState_STATE gil = PyGILState_Ensure();
  PyObject* module = PyImport_ImportModule("joyomni_ops._lib");
  PyObject* type = module ? PyObject_GetAttrString(module, "JoyError") : nullptr;
  PyErr_SetString(type ? type : PyExc_RuntimeError, joy_last_error());
  Py_XDECREF(type);
  Py_XDECREF(module);
  python_error error;
  error.persist();
  PyGILState_Release(gil);
  throw error;
}

int dtype_code(ScalarType t) { return t == at::kBFloat16 ? JOY_DTYPE_BF16 : t == at::kHalf ? JOY_DTYPE_FP16 : JOY_DTYPE_FP32; }

Tensor bytes_like(int64_t n, const Tensor& t) { return at::empty({n}, t.options().dtype(at::kByte)); }

// ---------------------------------------------------------------------------------- quantiser
void quant(const Tensor& input, const Tensor& output_q, const Tensor& output_s, int rounding) {
  const std::pair<const char*, const Tensor&> all[] = {
      {"input", input}, {"output_q", output_q}, {"output_s", output_s}};
  for (const auto& [name, t] : all) {
    TORCH_CHECK(t.is_cuda(), name, " must be a CUDA tensor");
    TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
  }
  TORCH_CHECK(input.dim() == 2, "input must be [M, K]");
  TORCH_CHECK(output_q.sizes() == input.sizes(), "output_q shape must match input");
  TORCH_CHECK(output_q.scalar_type() == at::kFloat8_e4m3fn, "output_q must be torch.float8_e4m3fn");
  TORCH_CHECK(output_s.scalar_type() == at::kFloat, "output_s must be float32");
  TORCH_CHECK(output_s.numel() == input.size(0), "output_s must contain one scale per row");
  TORCH_CHECK(input.device() == output_q.device() && input.device() == output_s.device(),
              "input and outputs must be on the same device");
  TORCH_CHECK(input.scalar_type() == at::kBFloat16 || input.scalar_type() == at::kHalf,
              "input must be bfloat16 or float16");
  c10::DeviceGuard guard(input.device());
  check_status(joy_per_token_quant_fp8(ptr(input), dtype_code(input.scalar_type()), ptr(output_q),
                                       (float*)ptr(output_s), input.size(0), input.size(1), rounding,
                                       stream_of(input)));
}

// the reference's gfx950 kernel rounds by reciprocal multiply (per_token_quant_fp8_rocm.hip:72-77)
void sgl_per_token_quant_fp8(const Tensor& input, const Tensor& output_q, const Tensor& output_s) {
  quant(input, output_q, output_s, JOY_QUANT_RECIPROCAL);
}

void per_token_quant_fp8(const Tensor& input, const Tensor& output_q, const Tensor& output_s, bool exact_division) {
  quant(input, output_q, output_s, exact_division ? JOY_QUANT_DIVIDE : JOY_QUANT_RECIPROCAL);
}

// --------------------------------------------------------------------------------------- GEMM
struct Mnk {
  int64_t M, N, K;
};

// checks of fp8_gemm.cu:1457-1487, and dense rows of both operands
Mnk scaled_mm_checks(const Tensor& mat_a, const Tensor& mat_b, const Tensor& scales_a, const Tensor& scales_b,
                     ScalarType out_dtype, const OptTensor& bias) {
  TORCH_CHECK(mat_a.is_cuda(), "mat_a must be a CUDA tensor");
  TORCH_CHECK(mat_b.is_cuda(), "mat_b must be a CUDA tensor");
  TORCH_CHECK(mat_a.dim() == 2, "mat_a must be a 2D tensor");
  TORCH_CHECK(mat_b.dim() == 2, "mat_b must be a 2D tensor");
  TORCH_CHECK(mat_a.stride(1) == 1, "mat_a must be a row major tensor");
  TORCH_CHECK(mat_b.stride(0) == 1, "mat_b must be a column major tensor");
  TORCH_CHECK(mat_a.size(1) == mat_b.size(0), "mat_a and mat_b shapes cannot be multiplied");
  TORCH_CHECK((mat_a.size(1) * mat_a.element_size()) % 16 == 0,
              "mat_a must be multiple of 16 bytes for memory alignment");
  TORCH_CHECK((mat_b.size(0) * mat_b.element_size()) % 16 == 0,
              "mat_b must be multiple of 16 bytes for memory alignment");
  TORCH_CHECK(mat_a.scalar_type() == at::kFloat8_e4m3fn, "mat_a must be Float8_e4m3fn");
  TORCH_CHECK(mat_b.scalar_type() == at::kFloat8_e4m3fn, "mat_b must be Float8_e4m3fn");
  TORCH_CHECK(out_dtype == at::kHalf || out_dtype == at::kBFloat16, "out_dtype must be Half or BFloat16");
  TORCH_CHECK(scales_a.numel() == mat_a.size(0), "size of scales_a is not matched");
  TORCH_CHECK(scales_b.numel() == mat_b.size(1), "size of scales_b is not matched");
  TORCH_CHECK(scales_a.is_contiguous(), "scales_a must be contiguous");
  TORCH_CHECK(scales_b.is_contiguous(), "scales_b msut be contiguous");
  TORCH_CHECK(scales_a.scalar_type() == at::kFloat, "scales_a must be Float32");
  TORCH_CHECK(scales_b.scalar_type() == at::kFloat, "scales_b must be Float32");
  const Mnk s = {mat_a.size(0), mat_b.size(1), mat_a.size(1)};
  if (bias) {
    TORCH_CHECK(bias->numel() == s.N, "size of bias is not matched");
    TORCH_CHECK(bias->is_contiguous(), "bias must be contiguous");
    TORCH_CHECK(bias->scalar_type() == out_dtype, "bias dtype must match output dtype");
  }
  TORCH_CHECK(s.M <= 1 || mat_a.stride(0) == s.K, "mat_a rows must be dense (stride(0) == K)");
  TORCH_CHECK(s.N <= 1 || mat_b.stride(1) == s.K, "mat_b columns must be dense (stride(1) == K)");
  TORCH_CHECK((s.N * 2) % 16 == 0, "out must be multiple of 16 bytes for memory alignment");
  return s;
}

// Split-K workspace of the small-M plans (undefined where the shape uses none), allocated from
// torch's caching allocator like the output, so a captured graph keeps its own.
Tensor gemm_workspace(const Mnk& s, const Tensor& like, int64_t* bytes) {
  *bytes = joy_fp8_scaled_mm_workspace_size(s.M, s.N, s.K);
  if (*bytes > 0) return bytes_like(*bytes, like);
  *bytes = 0;
  return Tensor();
}
void* ws_ptr(const Tensor& ws) { return ws.defined() ? ws.data_ptr() : nullptr; }

Tensor scaled_mm(const Tensor& mat_a, const Tensor& mat_b, const Tensor& scales_a, const Tensor& scales_b,
                 ScalarType out_dtype, const OptTensor& bias, int epilogue) {
  const Mnk s = scaled_mm_checks(mat_a, mat_b, scales_a, scales_b, out_dtype, bias);
  c10::DeviceGuard guard(mat_a.device());
  Tensor out = at::empty({s.M, s.N}, mat_a.options().dtype(out_dtype));
  int64_t bytes;
  const Tensor ws = gemm_workspace(s, mat_a, &bytes);
  check_status(joy_fp8_scaled_mm(ptr(mat_a), ptr(mat_b), (const float*)ptr(scales_a), (const float*)ptr(scales_b),
                                 ptr(bias), ptr(out), dtype_code(out_dtype), s.M, s.N, s.K, epilogue, ws_ptr(ws), bytes,
                                 stream_of(mat_a)));
  return out;
}

Tensor fp8_scaled_mm(const Tensor& mat_a, const Tensor& mat_b, const Tensor& scales_a, const Tensor& scales_b,
                     ScalarType out_dtype, const OptTensor& bias) {
  return scaled_mm(mat_a, mat_b, scales_a, scales_b, out_dtype, bias, JOY_EPILOGUE_NONE);
}

Tensor fp8_scaled_mm_gelu_tanh(const Tensor& mat_a, const Tensor& mat_b, const Tensor& scales_a,
                               const Tensor& scales_b, ScalarType out_dtype, const OptTensor& bias) {
  return scaled_mm(mat_a, mat_b, scales_a, scales_b, out_dtype, bias, JOY_EPILOGUE_GELU_TANH);
}

// out = residual + fp8_scaled_mm(...) * gate (fused_add_gate, sgl_fused_ops.py:302-305)
void gated_residual(const Tensor& mat_a, const Tensor& mat_b, const Tensor& scales_a, const Tensor& scales_b,
                    const Tensor& residual, const Tensor& gate_in, const OptTensor& bias, const Tensor& out) {
  const ScalarType out_dtype = residual.scalar_type();
  TORCH_CHECK(out_dtype == at::kHalf || out_dtype == at::kBFloat16, "residual must be Half or BFloat16");
  const Mnk s = scaled_mm_checks(mat_a, mat_b, scales_a, scales_b, out_dtype, bias);
  TORCH_CHECK(residual.is_cuda() && gate_in.is_cuda(), "residual and gate must be CUDA tensors");
  TORCH_CHECK(residual.dim() == 2 && residual.size(0) == s.M && residual.size(1) == s.N, "residual must be [M, N]");
  TORCH_CHECK(residual.stride(1) == 1 || s.N <= 1, "residual rows must be contiguous");
  TORCH_CHECK(gate_in.numel() == s.N, "size of gate is not matched");
  TORCH_CHECK(gate_in.scalar_type() == out_dtype, "gate dtype must match residual dtype");
  c10::DeviceGuard guard(mat_a.device());
  Tensor gate = gate_in.reshape({s.N});
  if (gate.stride(0) != 1 || (uintptr_t)gate.data_ptr() % 16 != 0)
    gate = gate.clone(at::MemoryFormat::Contiguous);  // N values: a 16-byte aligned copy
  int64_t bytes;
  const Tensor ws = gemm_workspace(s, mat_a, &bytes);
  check_status(joy_fp8_scaled_mm_gated_residual(
      ptr(mat_a), ptr(mat_b), (const float*)ptr(scales_a), (const float*)ptr(scales_b), ptr(bias), ptr(residual),
      s.M > 1 ? residual.stride(0) : s.N, ptr(gate), ptr(out), dtype_code(out_dtype), s.M, s.N, s.K, ws_ptr(ws), bytes,
      stream_of(mat_a)));
}

Tensor fp8_scaled_mm_gated_residual(const Tensor& mat_a, const Tensor& mat_b, const Tensor& scales_a,
                                    const Tensor& scales_b, const Tensor& residual, const Tensor& gate,
                                    const OptTensor& bias) {
  Tensor out = at::empty(residual.sizes(), residual.options());
  gated_residual(mat_a, mat_b, scales_a, scales_b, residual, gate, bias, out);
  return out;
}

void fp8_scaled_mm_gated_residual_(const Tensor& mat_a, const Tensor& mat_b, const Tensor& scales_a,
                                   const Tensor& scales_b, const Tensor& residual, const Tensor& gate,
                                   const OptTensor& bias) {
  TORCH_CHECK(residual.is_contiguous(), "an in-place residual must be contiguous");
  gated_residual(mat_a, mat_b, scales_a, scales_b, residual, gate, bias, residual);
}

// ------------------------------------------------------------------------ q/k RMSNorm + RoPE
// checks of fused_qknorm_rope_3d_kernel.cu:285-310
void fused_qk_norm_rope_3d_paired(const Tensor& q, const Tensor& k, int64_t seq_len, int64_t num_heads, double eps,
                                  const Tensor& q_weight, const Tensor& k_weight, const Tensor& cos, const Tensor& sin,
                                  const OptTensor& k_pre_rope) {
  TORCH_CHECK(q.dim() == 3, "q must be 3D [batch, seq_len*num_heads, head_dim]");
  TORCH_CHECK(k.dim() == 3, "k must be 3D [batch, seq_len*num_heads, head_dim]");
  TORCH_CHECK(q.sizes() == k.sizes(), "q and k must have the same shape");
  TORCH_CHECK(q_weight.dim() == 1 && k_weight.dim() == 1, "weights must be 1D [head_dim]");
  TORCH_CHECK(cos.dim() == 2 && sin.dim() == 2, "cos/sin must be 2D [seq_len, head_dim/2]");
  check_input(q, "q", at::kBFloat16);
  check_input(k, "k", at::kBFloat16);
  check_input(q_weight, "q_weight", at::kBFloat16);
  check_input(k_weight, "k_weight", at::kBFloat16);
  check_input(cos, "cos", at::kBFloat16);
  check_input(sin, "sin", at::kBFloat16);
  const int64_t head_dim = q.size(2);
  TORCH_CHECK(q.size(1) == seq_len * num_heads, "q.size(1) must equal seq_len*num_heads");
  TORCH_CHECK(q_weight.size(0) == head_dim && k_weight.size(0) == head_dim, "weight size must match head_dim");
  TORCH_CHECK(cos.size(0) == seq_len && cos.size(1) == head_dim / 2, "cos shape must be [seq_len, head_dim/2]");
  TORCH_CHECK(sin.size(0) == seq_len && sin.size(1) == head_dim / 2, "sin shape must be [seq_len, head_dim/2]");
  if (k_pre_rope) {
    TORCH_CHECK(k_pre_rope->sizes() == k.sizes(), "k_pre_rope must have the same shape as k");
    check_input(*k_pre_rope, "k_pre_rope", at::kBFloat16);
  }
  c10::DeviceGuard guard(q.device());
  check_status(joy_fused_qk_norm_rope_3d_paired(ptr(q), ptr(k), q.size(0), seq_len, num_heads, head_dim, (float)eps,
                                                ptr(q_weight), ptr(k_weight), ptr(cos), ptr(sin), ptr(k_pre_rope),
                                                stream_of(q)));
}

// Token stride of an output view of L tokens: [L, H, D], [1, L, H, D] or [L, H*D], dense heads. The
// kernel writes exactly L token rows through it, so a view with another token count (a short or
// mis-sliced output) is rejected before anything is launched.
int64_t token_stride(const OptTensor& o, int64_t L, int64_t H, int64_t D, const char* name, c10::Device device) {
  if (!o) return 0;
  const Tensor& t = *o;
  TORCH_CHECK(t.is_cuda() && t.device() == device, name, " must be a CUDA tensor on the device of qkv");
  TORCH_CHECK(t.scalar_type() == at::kBFloat16, name, " must be a bf16 CUDA tensor");
  int64_t d = 0;  // the token dimension
  if (t.dim() == 4) {
    TORCH_CHECK(t.size(0) == 1, name, " batch must be 1");
    d = 1;
  }
  if (t.dim() == 2) {
    TORCH_CHECK(t.size(1) == H * D && t.stride(1) == 1, name, " must have dense rows of H*D");
  } else {
    TORCH_CHECK(t.dim() - d == 3 && t.size(d + 1) == H && t.size(d + 2) == D, name, " must be [L, H, D]");
    TORCH_CHECK(t.stride(d + 2) == 1 && t.stride(d + 1) == D, name, " must have dense heads");
  }
  TORCH_CHECK(t.size(d) == L, name, " holds ", t.size(d), " tokens, expected ", L, " (the rows of qkv)");
  return L > 1 ? t.stride(d) : H * D;
}

// The norm/RoPE/ring outputs shared by fused_qkv_norm_rope_cache and fp8_qkv_norm_rope_cache.
struct RopeOutputs {
  int64_t q_stride, k_stride, v_stride, slots, capacity, cache_tokens;
};

RopeOutputs rope_output_checks(int64_t L, int64_t H, int64_t D, c10::Device device, const Tensor& q_weight,
                               const Tensor& k_weight, const Tensor& cos, const Tensor& sin, const OptTensor& q_out,
                               const OptTensor& k_out, const OptTensor& cache_k, const OptTensor& cache_v,
                               const OptTensor& v_out, int64_t cache_tokens) {
  const std::pair<const char*, const Tensor&> tables[] = {
      {"q_weight", q_weight}, {"k_weight", k_weight}, {"cos", cos}, {"sin", sin}};
  for (const auto& [name, t] : tables) {
    check_input(t, name, at::kBFloat16);
    TORCH_CHECK(t.device() == device, name, " must be on the device of qkv");
  }
  TORCH_CHECK(q_weight.numel() == D && k_weight.numel() == D, "weight size must match head_dim");
  TORCH_CHECK(cos.dim() == 2 && cos.size(0) == L && cos.size(1) == D / 2 && sin.sizes() == cos.sizes(),
              "cos/sin shape must be [seq_len, head_dim/2]");
  RopeOutputs r;
  r.q_stride = token_stride(q_out, L, H, D, "q_out", device);
  r.k_stride = token_stride(k_out, L, H, D, "k_out", device);
  r.v_stride = token_stride(v_out, L, H, D, "v_out", device);
  r.slots = r.capacity = 0;
  TORCH_CHECK(cache_k.has_value() == cache_v.has_value(), "cache_k and cache_v must be provided together");
  r.cache_tokens = cache_tokens < 0 ? L : cache_tokens;
  if (cache_k) {
    const std::pair<const char*, const Tensor&> ring[] = {{"cache_k", *cache_k}, {"cache_v", *cache_v}};
    for (const auto& [name, t] : ring)
      TORCH_CHECK(t.is_cuda() && t.device() == device && t.scalar_type() == at::kBFloat16, name,
                  " must be a bf16 CUDA tensor on the device of qkv");
    TORCH_CHECK(cache_k->is_contiguous() && cache_v->is_contiguous(), "cache_k/cache_v must be contiguous");
    TORCH_CHECK(cache_k->dim() == 4 && cache_k->sizes() == cache_v->sizes() && cache_k->size(2) == H &&
                    cache_k->size(3) == D,
                "cache must be [num_slots, capacity, H, D]");
    r.slots = cache_k->size(0);
    r.capacity = cache_k->size(1);
  }
  return r;
}

void fused_qkv_norm_rope_cache(const Tensor& qkv, int64_t num_heads, double eps, const Tensor& q_weight,
                               const Tensor& k_weight, const Tensor& cos, const Tensor& sin, const OptTensor& q_out,
                               const OptTensor& k_out, const OptTensor& cache_k, const OptTensor& cache_v, int64_t slot,
                               int64_t slot_offset, const OptTensor& v_out, int64_t cache_tokens,
                               bool cache_pre_rope) {
  TORCH_CHECK(qkv.is_cuda(), "qkv must be a CUDA tensor");
  TORCH_CHECK(qkv.scalar_type() == at::kBFloat16, "qkv dtype is ", dtype_name(qkv.scalar_type()),
              ", expected torch.bfloat16");
  TORCH_CHECK(qkv.dim() == 2 || (qkv.dim() == 3 && qkv.size(0) == 1), "qkv must be [L, 3*H*D] or [1, L, 3*H*D]");
  const int64_t d = qkv.dim() - 2;
  TORCH_CHECK(qkv.stride(d + 1) == 1, "qkv rows must be contiguous");
  const int64_t L = qkv.size(d), E3 = qkv.size(d + 1), H = num_heads;
  TORCH_CHECK(H > 0 && E3 % (3 * H) == 0, "qkv width must be 3*num_heads*head_dim");
  const int64_t D = E3 / (3 * H);
  const RopeOutputs r = rope_output_checks(L, H, D, qkv.device(), q_weight, k_weight, cos, sin, q_out, k_out, cache_k,
                                           cache_v, v_out, cache_tokens);
  c10::DeviceGuard guard(qkv.device());
  check_status(joy_fused_qkv_norm_rope_cache(
      ptr(qkv), L > 1 ? qkv.stride(d) : E3, L, H, D, (float)eps, ptr(q_weight), ptr(k_weight), ptr(cos), ptr(sin),
      ptr(q_out), r.q_stride, ptr(k_out), r.k_stride, ptr(v_out), r.v_stride, ptr(cache_k), ptr(cache_v), r.slots,
      r.capacity, slot, slot_offset, r.cache_tokens, cache_pre_rope ? 0 : 1, stream_of(qkv)));
}

void fp8_qkv_norm_rope_cache(const Tensor& mat_a, const Tensor& mat_b, const Tensor& scales_a, const Tensor& scales_b,
                             const OptTensor& bias, int64_t num_heads, double eps, const Tensor& q_weight,
                             const Tensor& k_weight, const Tensor& cos_in, const Tensor& sin_in, const OptTensor& q_out,
                             const OptTensor& k_out, const OptTensor& cache_k, const OptTensor& cache_v, int64_t slot,
                             int64_t slot_offset, const OptTensor& v_out, int64_t cache_tokens, bool cache_pre_rope) {
  const Mnk s = scaled_mm_checks(mat_a, mat_b, scales_a, scales_b, at::kBFloat16, bias);
  const int64_t H = num_heads;
  TORCH_CHECK(H > 0 && s.N % (3 * H) == 0, "mat_b width must be 3*num_heads*head_dim");
  const int64_t D = s.N / (3 * H);
  const RopeOutputs r = rope_output_checks(s.M, H, D, mat_a.device(), q_weight, k_weight, cos_in, sin_in, q_out, k_out,
                                           cache_k, cache_v, v_out, cache_tokens);
  c10::DeviceGuard guard(mat_a.device());
  // the fused epilogue reads the tables 16 bytes at a time: an aligned copy of a misaligned view
  const Tensor cos = (uintptr_t)cos_in.data_ptr() % 16 == 0 ? cos_in : cos_in.clone();
  const Tensor sin = (uintptr_t)sin_in.data_ptr() % 16 == 0 ? sin_in : sin_in.clone();
  int64_t bytes = joy_fp8_qkv_norm_rope_cache_scratch_size(s.M, s.K, H, D);
  // outputs whose byte offsets pass 2^31 take the unfused path, through an [M, N] bf16 buffer
  const std::pair<const OptTensor&, int64_t> outs[] = {{q_out, r.q_stride}, {k_out, r.k_stride}, {v_out, r.v_stride}};
  for (const auto& [t, stride] : outs)
    if (t && (s.M * stride + H * D) * 2 > 0x7fffffffLL) bytes = std::max(bytes, s.M * s.N * 2);
  // the tiles that do not take the fused epilogue pass through this [M, N] bf16 buffer (and the workspace after it)
  const Tensor scratch = bytes > 0 ? bytes_like(bytes, mat_a) : Tensor();
  check_status(joy_fp8_qkv_norm_rope_cache(
      ptr(mat_a), ptr(mat_b), (const float*)ptr(scales_a), (const float*)ptr(scales_b), ptr(bias), s.M, s.K, H, D,
      (float)eps, ptr(q_weight), ptr(k_weight), ptr(cos), ptr(sin), ptr(q_out), r.q_stride, ptr(k_out), r.k_stride,
      ptr(v_out), r.v_stride, ptr(cache_k), ptr(cache_v), r.slots, r.capacity, slot, slot_offset, r.cache_tokens,
      cache_pre_rope ? 0 : 1, ws_ptr(scratch), bytes, stream_of(mat_a)));
}

// ------------------------------------------------------------------------------ attention core
joy_bf16_view view_of(const Tensor& t, int64_t batch = 0) {  // of [B, L, H, D]
  return {(const char*)t.data_ptr() + batch * t.stride(0) * t.element_size(), t.size(1), t.stride(1), t.stride(2)};
}
// an optional view: null where the tensor is absent
struct OptView {
  joy_bf16_view v;
  const joy_bf16_view* p;
  explicit OptView(const OptTensor& t) : v{}, p(nullptr) {
    if (t) {
      v = view_of(*t);
      p = &v;
    }
  }
  OptView(const OptView&) = delete;
};

void attention(const Tensor& query, const Tensor& key, const Tensor& value, const Tensor& out,
               std::optional<double> scale) {
  const std::pair<const char*, const Tensor&> all[] = {{"query", query}, {"key", key}, {"value", value}, {"out", out}};
  for (const auto& [name, t] : all) {
    TORCH_CHECK(t.is_cuda(), name, " must be a CUDA tensor");
    TORCH_CHECK(t.dim() == 4, name, " must be [B, S, H, D]");
    TORCH_CHECK(t.scalar_type() == at::kBFloat16, name, " must be bfloat16");
    TORCH_CHECK(t.stride(3) == 1 || t.size(3) <= 1, name, " last dimension must be contiguous");
  }
  const int64_t B = query.size(0), Lq = query.size(1), H = query.size(2), D = query.size(3);
  TORCH_CHECK(key.sizes() == value.sizes(), "key and value must have the same shape");
  TORCH_CHECK(key.size(0) == B && key.size(2) == H && key.size(3) == D,
              "query, key and value must agree in batch, heads and head_dim");
  TORCH_CHECK(out.sizes() == query.sizes(), "out must have the shape of query");
  TORCH_CHECK(out.stride(2) == D, "out heads must be dense (stride(2) == head_dim)");
  const double sc = scale ? *scale : 1.0 / std::sqrt((double)D);
  c10::DeviceGuard guard(query.device());
  // fp32 parts of the key split (0 bytes where the call is not split), shared by the batches, which
  // follow each other on one stream
  const int64_t bytes = D == 128 ? joy_attention_workspace_size(Lq, key.size(1), H) : 0;
  const Tensor ws = bytes > 0 ? bytes_like(bytes, query) : Tensor();
  for (int64_t b = 0; b < B; ++b) {
    const joy_bf16_view q = view_of(query, b), k = view_of(key, b), v = view_of(value, b);
    check_status(joy_attention_fwd_workspace(&q, &k, &v, (char*)out.data_ptr() + b * out.stride(0) * 2, out.stride(1),
                                             H, D, (float)sc, ws_ptr(ws), bytes, stream_of(query)));
  }
}

Tensor sdpa_attention(const Tensor& query, const Tensor& key, const Tensor& value, std::optional<double> scale) {
  Tensor out = at::empty(query.sizes(), query.options());
  attention(query, key, value, out, scale);
  return out;
}

void sdpa_attention_out(const Tensor& query, const Tensor& key, const Tensor& value, const Tensor& out,
                        std::optional<double> scale) {
  attention(query, key, value, out, scale);
}

// ------------------------------------- cache read side: joint Q/K/V pack and cached-K rotation
// check_qkv_tensor of fused_joint_qkv_pack.cu:222-229
void check_qkv(const Tensor& t, const char* name, int64_t batch, int64_t heads, int64_t head_dim) {
  TORCH_CHECK(t.is_cuda(), name, " must be a CUDA tensor");
  TORCH_CHECK(t.scalar_type() == at::kBFloat16, name, " must be bfloat16");
  TORCH_CHECK(t.dim() == 4, name, " must be [B,L,H,D]");
  TORCH_CHECK(t.size(0) == batch && t.size(2) == heads && t.size(3) == head_dim, name, " has incompatible shape ",
              t.sizes());
  TORCH_CHECK(t.stride(3) == 1, name, " last dimension must be contiguous");
}

// checks of fused_joint_qkv_pack.cu:244-284
std::tuple<Tensor, Tensor, Tensor> fused_joint_qkv_pack(const Tensor& img_q, const Tensor& img_k, const Tensor& img_v,
                                                        const Tensor& txt_q, const Tensor& txt_k, const Tensor& txt_v,
                                                        const OptTensor& cached_k, const OptTensor& cached_v,
                                                        const Tensor& txt_q_weight, const Tensor& txt_k_weight,
                                                        double eps) {
  TORCH_CHECK(img_q.dim() == 4, "img_q must be [B,L,H,D]");
  const int64_t batch = img_q.size(0), img_len = img_q.size(1), heads = img_q.size(2), head_dim = img_q.size(3);
  TORCH_CHECK(batch == 1, "fused_joint_qkv_pack fast path requires batch=1");
  TORCH_CHECK(head_dim == 128, "fused_joint_qkv_pack requires head_dim=128");
  TORCH_CHECK(img_len > 0 && heads > 0, "image length and heads must be positive");
  check_qkv(img_q, "img_q", batch, heads, head_dim);
  check_qkv(img_k, "img_k", batch, heads, head_dim);
  check_qkv(img_v, "img_v", batch, heads, head_dim);
  TORCH_CHECK(img_k.size(1) == img_len && img_v.size(1) == img_len, "image Q/K/V lengths must match");
  const int64_t txt_len = txt_q.dim() == 4 ? txt_q.size(1) : 0;
  check_qkv(txt_q, "txt_q", batch, heads, head_dim);
  check_qkv(txt_k, "txt_k", batch, heads, head_dim);
  check_qkv(txt_v, "txt_v", batch, heads, head_dim);
  TORCH_CHECK(txt_len > 0 && txt_k.size(1) == txt_len && txt_v.size(1) == txt_len,
              "text Q/K/V lengths must match and be positive");
  check_input(txt_q_weight, "txt_q_weight", at::kBFloat16);
  check_input(txt_k_weight, "txt_k_weight", at::kBFloat16);
  TORCH_CHECK(txt_q_weight.dim() == 1 && txt_q_weight.numel() == head_dim, "txt_q_weight must be [head_dim]");
  TORCH_CHECK(txt_k_weight.dim() == 1 && txt_k_weight.numel() == head_dim, "txt_k_weight must be [head_dim]");
  TORCH_CHECK(cached_k.has_value() == cached_v.has_value(),
              "cached_k and cached_v must either both be present or both be absent");
  int64_t cache_len = 0;
  if (cached_k) {
    check_qkv(*cached_k, "cached_k", batch, heads, head_dim);
    check_qkv(*cached_v, "cached_v", batch, heads, head_dim);
    cache_len = cached_k->size(1);
    TORCH_CHECK(cached_v->size(1) == cache_len, "cached K/V lengths must match");
  }
  c10::DeviceGuard guard(img_q.device());
  Tensor out_q = at::empty({batch, img_len + txt_len, heads, head_dim}, img_q.options());
  Tensor out_k = at::empty({batch, cache_len + img_len + txt_len, heads, head_dim}, img_q.options());
  Tensor out_v = at::empty_like(out_k);
  const joy_bf16_view iq = view_of(img_q), ik = view_of(img_k), iv = view_of(img_v);
  const joy_bf16_view tq = view_of(txt_q), tk = view_of(txt_k), tv = view_of(txt_v);
  const OptView ck(cached_k), cv(cached_v);
  check_status(joy_fused_joint_qkv_pack(&iq, &ik, &iv, &tq, &tk, &tv, ck.p, cv.p, ptr(txt_q_weight), ptr(txt_k_weight),
                                        (float)eps, heads, head_dim, ptr(out_q), ptr(out_k), ptr(out_v),
                                        stream_of(img_q)));
  return {out_q, out_k, out_v};
}

// checks of fused_joint_qkv_pack.cu:351-381; the total length of the cached segments
int64_t cached_pack_checks(const Tensor& key0, const Tensor& value0, const OptTensor& key1, const OptTensor& value1,
                           const Tensor& cos, const Tensor& sin) {
  TORCH_CHECK(key0.dim() == 4, "key0 must be [B,L,H,D]");
  const int64_t batch = key0.size(0), len0 = key0.size(1), heads = key0.size(2), head_dim = key0.size(3);
  TORCH_CHECK(batch == 1, "fused_cached_kv_pack requires batch=1");
  TORCH_CHECK(head_dim == 128, "fused_cached_kv_pack requires head_dim=128");
  TORCH_CHECK(len0 > 0 && heads > 0, "cache length and heads must be positive");
  check_qkv(key0, "key0", batch, heads, head_dim);
  check_qkv(value0, "value0", batch, heads, head_dim);
  TORCH_CHECK(value0.size(1) == len0, "key0/value0 lengths must match");
  TORCH_CHECK(key1.has_value() == value1.has_value(),
              "key1 and value1 must either both be present or both be absent");
  int64_t len1 = 0;
  if (key1) {
    check_qkv(*key1, "key1", batch, heads, head_dim);
    check_qkv(*value1, "value1", batch, heads, head_dim);
    len1 = key1->size(1);
    TORCH_CHECK(len1 > 0 && value1->size(1) == len1, "key1/value1 lengths must match and be positive");
  }
  check_input(cos, "cos", at::kFloat);
  check_input(sin, "sin", at::kFloat);
  TORCH_CHECK(cos.sizes() == sin.sizes(), "cos/sin shapes must match");
  TORCH_CHECK(cos.numel() == (len0 + len1) * head_dim, "cos/sin must contain [total_cache_len, head_dim], got ",
              cos.sizes());
  return len0 + len1;
}

void cached_pack_launch(const Tensor& key0, const Tensor& value0, const OptTensor& key1, const OptTensor& value1,
                        const Tensor& cos, const Tensor& sin, const Tensor& out_k, const Tensor& out_v) {
  const joy_bf16_view k0 = view_of(key0), v0 = view_of(value0);
  const OptView k1(key1), v1(value1);
  c10::DeviceGuard guard(key0.device());
  check_status(joy_fused_cached_kv_pack(&k0, &v0, k1.p, v1.p, (const float*)ptr(cos), (const float*)ptr(sin),
                                        key0.size(2), key0.size(3), ptr(out_k), ptr(out_v), stream_of(key0)));
}

std::tuple<Tensor, Tensor> fused_cached_kv_pack(const Tensor& key0, const Tensor& value0, const OptTensor& key1,
                                                const OptTensor& value1, const Tensor& cos, const Tensor& sin) {
  const int64_t total = cached_pack_checks(key0, value0, key1, value1, cos, sin);
  Tensor out_k = at::empty({1, total, key0.size(2), key0.size(3)}, key0.options());
  Tensor out_v = at::empty_like(out_k);
  cached_pack_launch(key0, value0, key1, value1, cos, sin, out_k, out_v);
  return {out_k, out_v};
}

// a caller-provided pack output: bf16 CUDA [1, length, H, D] (or [length, H, D]), contiguous
void check_dense_out(const Tensor& t, const char* name, int64_t length, int64_t heads, int64_t head_dim) {
  TORCH_CHECK(t.is_cuda() && t.scalar_type() == at::kBFloat16, name, " must be a bf16 CUDA tensor");
  TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
  const int64_t d = t.dim() == 4 ? 1 : 0;
  TORCH_CHECK((t.dim() == 3 || (t.dim() == 4 && t.size(0) == 1)) && t.size(d) == length && t.size(d + 1) == heads &&
                  t.size(d + 2) == head_dim,
              name, " must be [1, ", length, ", ", heads, ", ", head_dim, "], got ", t.sizes());
}

void fused_cached_kv_pack_out(const Tensor& key0, const Tensor& value0, const OptTensor& key1, const OptTensor& value1,
                              const Tensor& cos, const Tensor& sin, const Tensor& out_k, const Tensor& out_v) {
  const int64_t total = cached_pack_checks(key0, value0, key1, value1, cos, sin);
  check_dense_out(out_k, "out_k", total, key0.size(2), key0.size(3));
  check_dense_out(out_v, "out_v", total, key0.size(2), key0.size(3));
  cached_pack_launch(key0, value0, key1, value1, cos, sin, out_k, out_v);
}

void fused_text_qkv_pack(const Tensor& txt_q, const Tensor& txt_k, const Tensor& txt_v, const Tensor& txt_q_weight,
                         const Tensor& txt_k_weight, double eps, const Tensor& out_q, const Tensor& out_k,
                         const Tensor& out_v) {
  TORCH_CHECK(txt_q.dim() == 4, "txt_q must be [B,L,H,D]");
  const int64_t batch = txt_q.size(0), txt_len = txt_q.size(1), heads = txt_q.size(2), head_dim = txt_q.size(3);
  TORCH_CHECK(batch == 1, "fused_text_qkv_pack requires batch=1");
  TORCH_CHECK(head_dim == 128, "fused_text_qkv_pack requires head_dim=128");
  check_qkv(txt_q, "txt_q", batch, heads, head_dim);
  check_qkv(txt_k, "txt_k", batch, heads, head_dim);
  check_qkv(txt_v, "txt_v", batch, heads, head_dim);
  TORCH_CHECK(txt_len > 0 && heads > 0 && txt_k.size(1) == txt_len && txt_v.size(1) == txt_len,
              "text Q/K/V lengths must match and be positive");
  const std::pair<const char*, const Tensor&> weights[] = {{"txt_q_weight", txt_q_weight},
                                                           {"txt_k_weight", txt_k_weight}};
  for (const auto& [name, t] : weights) {
    check_input(t, name, at::kBFloat16);
    TORCH_CHECK(t.dim() == 1 && t.numel() == head_dim, name, " must be [head_dim]");
  }
  check_dense_out(out_q, "out_q", txt_len, heads, head_dim);
  check_dense_out(out_k, "out_k", txt_len, heads, head_dim);
  check_dense_out(out_v, "out_v", txt_len, heads, head_dim);
  const joy_bf16_view q = view_of(txt_q), k = view_of(txt_k), v = view_of(txt_v);
  c10::DeviceGuard guard(txt_q.device());
  check_status(joy_fused_text_qkv_pack(&q, &k, &v, ptr(txt_q_weight), ptr(txt_k_weight), (float)eps, heads, head_dim,
                                       ptr(out_q), ptr(out_k), ptr(out_v), stream_of(txt_q)));
}

// ------------------------------------------------------------------ adaLN norm and modulation
struct NormArgs {
  int64_t M, N;
  Tensor gamma, beta, scale, shift;  // gamma, beta undefined where absent
};

// checks of fused_norm_scale_shift.cu:240-262
NormArgs norm_args(const Tensor& x, const OptTensor& gamma, const OptTensor& beta, const Tensor& scale,
                   const Tensor& shift, int64_t norm_type) {
  TORCH_CHECK(x.is_cuda(), "x must be a CUDA tensor");
  TORCH_CHECK(scale.is_cuda(), "scale must be a CUDA tensor");
  TORCH_CHECK(shift.is_cuda(), "shift must be a CUDA tensor");
  TORCH_CHECK(x.dim() == 2, "x must be 2D [M, N]");
  TORCH_CHECK(x.stride(1) == 1, "x last dim must be contiguous");
  NormArgs a;
  a.M = x.size(0);
  a.N = x.size(1);
  TORCH_CHECK(a.N % 4 == 0, "N must be divisible by 4");
  TORCH_CHECK(scale.dim() == 2 && shift.dim() == 2, "scale/shift must be 2D [M, N] or [1, N]");
  TORCH_CHECK(scale.size(0) == shift.size(0), "scale/shift row counts must match");
  TORCH_CHECK(scale.size(0) == 1 || scale.size(0) == a.M,
              "scale/shift rows must be 1 (broadcast) or M (per-row modulation)");
  TORCH_CHECK(scale.size(1) == a.N && shift.size(1) == a.N, "scale/shift last dim must be N");
  TORCH_CHECK(scale.stride(1) == 1 && shift.stride(1) == 1, "scale/shift last dim must be contiguous");
  const ScalarType t = x.scalar_type();
  TORCH_CHECK(t == scale.scalar_type() && t == shift.scalar_type(), "x/scale/shift dtype must match");
  TORCH_CHECK(norm_type == 0 || norm_type == 1, "norm_type must be 0 (layer) or 1 (rms)");
  TORCH_CHECK(t == at::kBFloat16 || t == at::kHalf || t == at::kFloat,
              "Unsupported dtype; use float32/float16/bfloat16");
  if (gamma) {
    TORCH_CHECK(gamma->numel() == a.N, "gamma must be length N");
    a.gamma = gamma->to(t).contiguous();
  }
  if (beta) {
    TORCH_CHECK(beta->numel() == a.N, "beta must be length N");
    a.beta = beta->to(t).contiguous();
  }
  // the kernel reads scale/shift rows densely, as the reference kernel does (:112-117)
  a.scale = scale.contiguous();
  a.shift = shift.contiguous();
  return a;
}

Tensor fused_norm_scale_shift(const Tensor& x, const OptTensor& gamma, const OptTensor& beta, const Tensor& scale,
                              const Tensor& shift, int64_t norm_type, double eps) {
  const NormArgs a = norm_args(x, gamma, beta, scale, shift, norm_type);
  c10::DeviceGuard guard(x.device());
  Tensor y = at::empty({a.M, a.N}, x.options());
  check_status(joy_fused_norm_scale_shift(ptr(x), a.M > 1 ? x.stride(0) : a.N, dtype_code(x.scalar_type()),
                                          ws_ptr(a.gamma), ws_ptr(a.beta), ptr(a.scale), ptr(a.shift), a.scale.size(0),
                                          ptr(y), a.M, a.N, (int)norm_type, (float)eps, stream_of(x)));
  return y;
}

void fused_norm_scale_shift_fp8(const Tensor& x, const OptTensor& gamma, const OptTensor& beta, const Tensor& scale,
                                const Tensor& shift, int64_t norm_type, double eps, const Tensor& output_q,
                                const Tensor& output_s, const OptTensor& out, bool exact_division) {
  const NormArgs a = norm_args(x, gamma, beta, scale, shift, norm_type);
  const ScalarType t = x.scalar_type();
  TORCH_CHECK(t == at::kBFloat16 || t == at::kHalf, "x must be bfloat16 or float16");
  TORCH_CHECK(output_q.is_cuda() && output_q.is_contiguous() && output_q.scalar_type() == at::kFloat8_e4m3fn &&
                  output_q.dim() == 2 && output_q.size(0) == a.M && output_q.size(1) == a.N,
              "output_q must be a contiguous float8_e4m3fn [M, N] CUDA tensor");
  TORCH_CHECK(output_s.is_cuda() && output_s.is_contiguous() && output_s.scalar_type() == at::kFloat &&
                  output_s.numel() == a.M,
              "output_s must contain one float32 scale per row");
  if (out)
    TORCH_CHECK(out->is_cuda() && out->is_contiguous() && out->scalar_type() == t && out->dim() == 2 &&
                    out->size(0) == a.M && out->size(1) == a.N,
                "out must be a contiguous [M, N] CUDA tensor of x's dtype");
  c10::DeviceGuard guard(x.device());
  check_status(joy_fused_norm_scale_shift_fp8(
      ptr(x), a.M > 1 ? x.stride(0) : a.N, dtype_code(t), ws_ptr(a.gamma), ws_ptr(a.beta), ptr(a.scale), ptr(a.shift),
      a.scale.size(0), ptr(out), ptr(output_q), (float*)ptr(output_s),
      exact_division ? JOY_QUANT_DIVIDE : JOY_QUANT_RECIPROCAL, a.M, a.N, (int)norm_type, (float)eps, stream_of(x)));
}

}  // namespace

// The C ABI that these operators were compiled for: compared by the package when it has loaded the library (an
// exception during the load itself would end the process).
extern "C" __attribute__((visibility("default"))) int joy_torch_abi_version(void) { return JOY_ABI_VERSION; }

TORCH_LIBRARY_IMPL(joyomni_ops, CUDA, m) {
  m.impl("sgl_per_token_quant_fp8", sgl_per_token_quant_fp8);
  m.impl("per_token_quant_fp8", per_token_quant_fp8);
  m.impl("fp8_scaled_mm", fp8_scaled_mm);
  m.impl("fp8_scaled_mm_gelu_tanh", fp8_scaled_mm_gelu_tanh);
  m.impl("fp8_scaled_mm_gated_residual", fp8_scaled_mm_gated_residual);
  m.impl("fp8_scaled_mm_gated_residual_", fp8_scaled_mm_gated_residual_);
  m.impl("fused_qk_norm_rope_3d_paired", fused_qk_norm_rope_3d_paired);
  m.impl("fused_qkv_norm_rope_cache", fused_qkv_norm_rope_cache);
  m.impl("fp8_qkv_norm_rope_cache", fp8_qkv_norm_rope_cache);
  m.impl("sdpa_attention", sdpa_attention);
  m.impl("sdpa_attention_out", sdpa_attention_out);
  m.impl("fused_joint_qkv_pack", fused_joint_qkv_pack);
  m.impl("fused_cached_kv_pack", fused_cached_kv_pack);
  m.impl("fused_cached_kv_pack_out", fused_cached_kv_pack_out);
  m.impl("fused_text_qkv_pack", fused_text_qkv_pack);
  m.impl("fused_norm_scale_shift", fused_norm_scale_shift);
  m.impl("fused_norm_scale_shift_fp8", fused_norm_scale_shift_fp8);
}
