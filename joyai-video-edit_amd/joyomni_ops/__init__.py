"""joyomni_ops -- MI355X (gfx950) drop-in for the reference's operator package.

Same namespace, op schemas, FakeTensor registrations and Python wrappers as the
reference's ``joyomni_ops/joyomni_ops/__init__.py`` (schemas from
``joyomni_ops/csrc/pybind.cpp:52-75``), so ``torch.ops.joyomni_ops.*`` and
``from joyomni_ops import ...`` keep working for ``deploy/xvideo``.

The quantised hot path -- ``sgl_per_token_quant_fp8``, ``fp8_scaled_mm``,
``fused_qk_norm_rope_3d_paired``, the new ``fused_qkv_norm_rope_cache``, the
cache read side ``fused_joint_qkv_pack`` / ``fused_cached_kv_pack`` and the
adaLN ``fused_norm_scale_shift`` (plus its FP8-emitting variant) -- runs in
hand-written gfx950 kernels of ``libjoyomni_hip.so`` reached through its C ABI
(``include/joyomni_hip.h``); the operators' device implementations on top of it
are C++ (``csrc/torch_ops.cpp``, ``libjoyomni_torch.so``). Importing fails when
either library is missing, exactly like the reference (``__init__.py:15-19``);
nothing falls back.

``rmsnorm``, which the model never calls, keeps its reference schema as a
torch device composition, so the reference's imports
(``sgl_fused_ops.py:27-33``) still resolve.
"""
from __future__ import annotations

from typing import Optional

import torch

from . import _lib

_LIB = _lib.load()  # raises ImportError when the HIP library is not built

__all__ = [
    "fused_qk_norm_rope_3d_paired",
    "fused_joint_qkv_pack",
    "fused_cached_kv_pack",
    "fused_norm_scale_shift",
    "rmsnorm",
    "sgl_per_token_quant_fp8",
    "fp8_scaled_mm",
    "has_quant",
    "has_fp8",
    # additions of this build
    "per_token_quant_fp8",
    "fp8_scaled_mm_gelu_tanh",
    "fused_qkv_norm_rope_cache",
    "fp8_qkv_norm_rope_cache",
    "fused_norm_scale_shift_fp8",
    "fp8_scaled_mm_gated_residual",
    "fused_cached_kv_pack_out",
    "fused_text_qkv_pack",
    "sdpa_attention",
    "sdpa_attention_out",
]

_NS = "joyomni_ops"
_lib_def = torch.library.Library(_NS, "DEF")

# --- reference schemas (pybind.cpp:52-75); one annotation added: the kernel writes k_pre_rope
# (fused_qknorm_rope_3d_kernel.cu:97-100), which the reference schema leaves undeclared, so under
# torch.compile functionalisation would not see that write. Declaring it mutable keeps every call
# site valid and makes the write visible. ---
_lib_def.define(
    "fused_qk_norm_rope_3d_paired(Tensor! q, Tensor! k, int seq_len, int num_heads, float eps, "
    "Tensor q_weight, Tensor k_weight, Tensor cos, Tensor sin, Tensor(a!)? k_pre_rope) -> ()")
_lib_def.define(
    "fused_joint_qkv_pack(Tensor img_q, Tensor img_k, Tensor img_v, "
    "Tensor txt_q, Tensor txt_k, Tensor txt_v, Tensor? cached_k, Tensor? cached_v, "
    "Tensor txt_q_weight, Tensor txt_k_weight, float eps) -> (Tensor, Tensor, Tensor)")
_lib_def.define(
    "fused_cached_kv_pack(Tensor key0, Tensor value0, Tensor? key1, Tensor? value1, "
    "Tensor cos, Tensor sin) -> (Tensor, Tensor)")
_lib_def.define(
    "fused_norm_scale_shift(Tensor x, Tensor? gamma_opt, Tensor? beta_opt, "
    "Tensor scale, Tensor shift, int norm_type, float eps) -> Tensor")
_lib_def.define("rmsnorm(Tensor x, Tensor weight, float eps) -> Tensor")
_lib_def.define("sgl_per_token_quant_fp8(Tensor input, Tensor! output_q, Tensor! output_s) -> ()")
_lib_def.define(
    "fp8_scaled_mm(Tensor mat_a, Tensor mat_b, Tensor scales_a, Tensor scales_b, "
    "ScalarType out_dtype, Tensor? bias) -> Tensor")

# --- additions of this build ---
_lib_def.define(
    "per_token_quant_fp8(Tensor input, Tensor! output_q, Tensor! output_s, bool exact_division) -> ()")
_lib_def.define(
    "fp8_scaled_mm_gelu_tanh(Tensor mat_a, Tensor mat_b, Tensor scales_a, Tensor scales_b, "
    "ScalarType out_dtype, Tensor? bias) -> Tensor")
_lib_def.define(
    "fp8_scaled_mm_gated_residual(Tensor mat_a, Tensor mat_b, Tensor scales_a, Tensor scales_b, "
    "Tensor residual, Tensor gate, Tensor? bias) -> Tensor")
_lib_def.define(
    "fp8_scaled_mm_gated_residual_(Tensor mat_a, Tensor mat_b, Tensor scales_a, Tensor scales_b, "
    "Tensor(a!) residual, Tensor gate, Tensor? bias) -> ()")
_lib_def.define(
    "fused_norm_scale_shift_fp8(Tensor x, Tensor? gamma_opt, Tensor? beta_opt, Tensor scale, "
    "Tensor shift, int norm_type, float eps, Tensor(a!) output_q, Tensor(b!) output_s, "
    "Tensor(c!)? out, bool exact_division) -> ()")
_lib_def.define(
    "fused_qkv_norm_rope_cache(Tensor qkv, int num_heads, float eps, Tensor q_weight, "
    "Tensor k_weight, Tensor cos, Tensor sin, Tensor(a!)? q_out, Tensor(b!)? k_out, "
    "Tensor(c!)? cache_k, Tensor(d!)? cache_v, int slot, int slot_offset, Tensor(e!)? v_out=None, "
    "int cache_tokens=-1, bool cache_pre_rope=True) -> ()")
_lib_def.define(
    "fp8_qkv_norm_rope_cache(Tensor mat_a, Tensor mat_b, Tensor scales_a, Tensor scales_b, Tensor? bias, "
    "int num_heads, float eps, Tensor q_weight, Tensor k_weight, Tensor cos, Tensor sin, Tensor(a!)? q_out, "
    "Tensor(b!)? k_out, Tensor(c!)? cache_k, Tensor(d!)? cache_v, int slot, int slot_offset, "
    "Tensor(e!)? v_out=None, int cache_tokens=-1, bool cache_pre_rope=True) -> ()")
_lib_def.define(
    "fused_cached_kv_pack_out(Tensor key0, Tensor value0, Tensor? key1, Tensor? value1, "
    "Tensor cos, Tensor sin, Tensor(a!) out_k, Tensor(b!) out_v) -> ()")
_lib_def.define(
    "fused_text_qkv_pack(Tensor txt_q, Tensor txt_k, Tensor txt_v, Tensor txt_q_weight, "
    "Tensor txt_k_weight, float eps, Tensor(a!) out_q, Tensor(b!) out_k, Tensor(c!) out_v) -> ()")

_lib_def.define("sdpa_attention(Tensor query, Tensor key, Tensor value, float? scale=None) -> Tensor")
_lib_def.define(
    "sdpa_attention_out(Tensor query, Tensor key, Tensor value, Tensor(a!) out, float? scale=None) -> ()")

_ops = torch.ops.joyomni_ops


# The operators' device implementations: argument checks, allocation and the C-ABI call, in C++
# (csrc/torch_ops.cpp).
_lib.load_ops()


_DEVICE = torch._C.DispatchKeySet(torch._C.DispatchKey.CUDA)


def _quant_impl(input, output_q, output_s, rounding):
    """The quantiser's device implementation by C-ABI rounding code, called for tensors of any device
    (its own checks refuse the others)."""
    if rounding not in (_lib.JOY_QUANT_DIVIDE, _lib.JOY_QUANT_RECIPROCAL):
        raise _lib.JoyError("rounding must be JOY_QUANT_DIVIDE or JOY_QUANT_RECIPROCAL")
    _ops.per_token_quant_fp8.default.redispatch(_DEVICE, input, output_q, output_s,
                                                rounding == _lib.JOY_QUANT_DIVIDE)


def _scaled_mm_impl(mat_a, mat_b, scales_a, scales_b, out_dtype, bias, epilogue):
    """The GEMM's device implementation by C-ABI epilogue code, likewise."""
    op = {_lib.JOY_EPILOGUE_NONE: _ops.fp8_scaled_mm, _lib.JOY_EPILOGUE_GELU_TANH: _ops.fp8_scaled_mm_gelu_tanh}.get(epilogue)
    if op is None:
        raise _lib.JoyError(f"unknown epilogue {epilogue}")
    return op.default.redispatch(_DEVICE, mat_a, mat_b, scales_a, scales_b, out_dtype, bias)


# --------------------------------------------------------------------------
# rmsnorm: outside the quantised path (the model never calls it); a torch
# device composition of rmsnorm.cu:60-84 keeps the reference import working
# --------------------------------------------------------------------------
@torch.library.impl(_lib_def, "rmsnorm", "CUDA")
def _rmsnorm_cuda(x, weight, eps):
    xf = x.float()
    return ((xf * torch.rsqrt(xf.square().mean(-1, keepdim=True) + eps)) * weight.float()).to(x.dtype)


# --------------------------------------------------------------------------
# FakeTensor kernels (reference __init__.py:39-101) so torch.compile keeps the
# ops opaque inside one graph.
# --------------------------------------------------------------------------
@torch.library.register_fake("joyomni_ops::fused_qk_norm_rope_3d_paired")
def _fake_fused_qk_norm_rope_3d_paired(q, k, seq_len, num_heads, eps, q_weight, k_weight, cos,
                                       sin, k_pre_rope=None):
    return None


@torch.library.register_fake("joyomni_ops::fused_joint_qkv_pack")
def _fake_fused_joint_qkv_pack(img_q, img_k, img_v, txt_q, txt_k, txt_v, cached_k, cached_v,
                               txt_q_weight, txt_k_weight, eps):
    batch, img_len, heads, head_dim = img_q.shape
    txt_len = txt_q.shape[1]
    cache_len = cached_k.shape[1] if cached_k is not None else 0
    out_q = img_q.new_empty((batch, img_len + txt_len, heads, head_dim))
    out_k = img_q.new_empty((batch, cache_len + img_len + txt_len, heads, head_dim))
    return out_q, out_k, torch.empty_like(out_k)


@torch.library.register_fake("joyomni_ops::fused_cached_kv_pack")
def _fake_fused_cached_kv_pack(key0, value0, key1, value1, cos, sin):
    batch, len0, heads, head_dim = key0.shape
    len1 = key1.shape[1] if key1 is not None else 0
    out_key = key0.new_empty((batch, len0 + len1, heads, head_dim))
    return out_key, torch.empty_like(out_key)


@torch.library.register_fake("joyomni_ops::fused_norm_scale_shift")
def _fake_fused_norm_scale_shift(x, gamma, beta, scale, shift, norm_type, eps):
    return torch.empty_like(x)


@torch.library.register_fake("joyomni_ops::fused_norm_scale_shift_fp8")
def _fake_fused_norm_scale_shift_fp8(x, gamma, beta, scale, shift, norm_type, eps, output_q, output_s,
                                     out, exact_division):
    return None


@torch.library.register_fake("joyomni_ops::rmsnorm")
def _fake_rmsnorm(x, weight, eps):
    return torch.empty_like(x)


@torch.library.register_fake("joyomni_ops::sgl_per_token_quant_fp8")
def _fake_sgl_per_token_quant_fp8(input, output_q, output_s):
    return None


@torch.library.register_fake("joyomni_ops::per_token_quant_fp8")
def _fake_per_token_quant_fp8(input, output_q, output_s, exact_division):
    return None


@torch.library.register_fake("joyomni_ops::fp8_scaled_mm")
def _fake_fp8_scaled_mm(mat_a, mat_b, scales_a, scales_b, out_dtype, bias=None):
    return mat_a.new_empty((mat_a.shape[0], mat_b.shape[1]), dtype=out_dtype)


@torch.library.register_fake("joyomni_ops::fp8_scaled_mm_gelu_tanh")
def _fake_fp8_scaled_mm_gelu_tanh(mat_a, mat_b, scales_a, scales_b, out_dtype, bias=None):
    return mat_a.new_empty((mat_a.shape[0], mat_b.shape[1]), dtype=out_dtype)


@torch.library.register_fake("joyomni_ops::fp8_scaled_mm_gated_residual")
def _fake_fp8_scaled_mm_gated_residual(mat_a, mat_b, scales_a, scales_b, residual, gate, bias=None):
    return residual.new_empty(residual.shape)


@torch.library.register_fake("joyomni_ops::fp8_scaled_mm_gated_residual_")
def _fake_fp8_scaled_mm_gated_residual_inplace(mat_a, mat_b, scales_a, scales_b, residual, gate, bias=None):
    return None


@torch.library.register_fake("joyomni_ops::fused_qkv_norm_rope_cache")
def _fake_fused_qkv_norm_rope_cache(qkv, num_heads, eps, q_weight, k_weight, cos, sin, q_out,
                                    k_out, cache_k, cache_v, slot, slot_offset, v_out=None, cache_tokens=-1,
                                    cache_pre_rope=True):
    return None


@torch.library.register_fake("joyomni_ops::fp8_qkv_norm_rope_cache")
def _fake_fp8_qkv_norm_rope_cache(mat_a, mat_b, scales_a, scales_b, bias, num_heads, eps, q_weight, k_weight, cos,
                                  sin, q_out, k_out, cache_k, cache_v, slot, slot_offset, v_out=None,
                                  cache_tokens=-1, cache_pre_rope=True):
    return None


@torch.library.register_fake("joyomni_ops::fused_cached_kv_pack_out")
def _fake_fused_cached_kv_pack_out(key0, value0, key1, value1, cos, sin, out_k, out_v):
    return None


@torch.library.register_fake("joyomni_ops::sdpa_attention")
def _fake_sdpa_attention(query, key, value, scale=None):
    return query.new_empty(query.shape)


@torch.library.register_fake("joyomni_ops::sdpa_attention_out")
def _fake_sdpa_attention_out(query, key, value, out, scale=None):
    return None


@torch.library.register_fake("joyomni_ops::fused_text_qkv_pack")
def _fake_fused_text_qkv_pack(txt_q, txt_k, txt_v, txt_q_weight, txt_k_weight, eps, out_q, out_k, out_v):
    return None


# --------------------------------------------------------------------------
# Python wrappers with the reference's names and signatures (__init__.py:104-153)
# --------------------------------------------------------------------------
def fused_qk_norm_rope_3d_paired(q, k, seq_len, num_heads, eps, q_weight, k_weight, cos, sin,
                                 k_pre_rope=None):
    """Per-head RMSNorm then interleaved RoPE on q and k, written over them (bf16 [B, seq_len * num_heads,
    head_dim]); ``k_pre_rope`` optionally receives k after the norm and before the rotation."""
    _ops.fused_qk_norm_rope_3d_paired(q, k, seq_len, num_heads, eps, q_weight, k_weight, cos, sin,
                                      k_pre_rope)


def fused_joint_qkv_pack(img_q, img_k, img_v, txt_q, txt_k, txt_v, cached_k, cached_v,
                         txt_q_weight, txt_k_weight, eps=1e-6):
    """Joint attention operands in fresh tensors: Q = [image | normed text], K / V = [cache | image | text],
    the text q / k RMS-normalised with two roundings; batch 1, head_dim 128, bf16."""
    return _ops.fused_joint_qkv_pack(img_q, img_k, img_v, txt_q, txt_k, txt_v, cached_k, cached_v,
                                     txt_q_weight, txt_k_weight, eps)


def fused_cached_kv_pack(key0, value0, key1, value1, cos, sin):
    """Cached keys stored before RoPE (one or two segments) rotated with fp32 full-width tables and
    concatenated, values concatenated alongside; batch 1, head_dim 128, bf16."""
    return _ops.fused_cached_kv_pack(key0, value0, key1, value1, cos, sin)


def fused_norm_scale_shift(x, gamma, beta, scale, shift, norm_type, eps=1e-5):
    """LayerNorm or RMSNorm of each row of x (optional affine gamma / beta), then adaLN modulation
    ``* (1 + scale) + shift``; ``norm_type`` is ``"layer"`` or ``"rms"``."""
    nt = 0 if norm_type == "layer" else 1 if norm_type == "rms" else -1
    return _ops.fused_norm_scale_shift(x, gamma, beta, scale, shift, nt, eps)


def fused_norm_scale_shift_fp8(x, gamma, beta, scale, shift, norm_type, eps, output_q, output_s,
                               out=None, exact_division: bool = True):
    """Norm + adaLN modulation quantised per token to e4m3fn in one pass: output_q/output_s are
    bit-identical to ``per_token_quant_fp8(fused_norm_scale_shift(...))``; ``out`` optionally
    receives the modulated row itself."""
    nt = 0 if norm_type == "layer" else 1 if norm_type == "rms" else -1
    _ops.fused_norm_scale_shift_fp8(x, gamma, beta, scale, shift, nt, eps, output_q, output_s, out,
                                    exact_division)


def rmsnorm(x, weight, eps=1e-6):
    """Row-wise RMS normalisation of x [M, N] scaled by weight [N]."""
    return _ops.rmsnorm(x, weight, eps)


def has_fp8() -> bool:
    return hasattr(_ops, "fp8_scaled_mm")


def has_quant() -> bool:
    return hasattr(_ops, "sgl_per_token_quant_fp8")


def sgl_per_token_quant_fp8(input, output_q, output_s):
    _ops.sgl_per_token_quant_fp8(input, output_q, output_s)


def fp8_scaled_mm(mat_a, mat_b, scales_a, scales_b, out_dtype, bias: Optional[torch.Tensor] = None):
    return _ops.fp8_scaled_mm(mat_a, mat_b, scales_a, scales_b, out_dtype, bias)


def per_token_quant_fp8(input, output_q, output_s, exact_division: bool = True):
    """Per-token e4m3fn quantisation; exact_division=True is bit-identical to
    ``_quantize_per_token_impl`` (deploy/xvideo/models/dit/fp8_linear.py:38-43)."""
    _ops.per_token_quant_fp8(input, output_q, output_s, exact_division)


def fp8_scaled_mm_gelu_tanh(mat_a, mat_b, scales_a, scales_b, out_dtype,
                            bias: Optional[torch.Tensor] = None):
    """fp8_scaled_mm followed by GELU-tanh on the rounded output, in one kernel."""
    return _ops.fp8_scaled_mm_gelu_tanh(mat_a, mat_b, scales_a, scales_b, out_dtype, bias)


def fp8_scaled_mm_gated_residual(mat_a, mat_b, scales_a, scales_b, residual, gate,
                                 bias: Optional[torch.Tensor] = None, inplace: bool = False):
    """residual + fp8_scaled_mm(mat_a, mat_b, ...) * gate in one kernel (the block's out-projection /
    FFN-down followed by fused_add_gate); output dtype = residual dtype, gate [N]. Bit-identical to
    ``torch.addcmul(residual, fp8_scaled_mm(...), gate)``. ``inplace=True`` writes into ``residual``
    (contiguous) and returns it."""
    if inplace:
        _ops.fp8_scaled_mm_gated_residual_(mat_a, mat_b, scales_a, scales_b, residual, gate, bias)
        return residual
    return _ops.fp8_scaled_mm_gated_residual(mat_a, mat_b, scales_a, scales_b, residual, gate, bias)


def fused_qkv_norm_rope_cache(qkv, num_heads, eps, q_weight, k_weight, cos, sin, q_out,
                              k_out=None, cache_k=None, cache_v=None, slot=0, slot_offset=0, v_out=None,
                              cache_tokens: int = -1, cache_pre_rope: bool = True):
    """QKV split + q/k RMSNorm + RoPE in one pass.

    Roped Q / K go to ``q_out`` / ``k_out`` (either may be None; without ``q_out`` Q is not read).
    The first ``cache_tokens`` tokens (all when negative; ``kv_cache_write_seq_len``) of K and V
    land in ring slot ``slot`` from row ``slot_offset``: K normalised before rotation when
    ``cache_pre_rope`` (``kv_cache_pre_rope=True``), else rotated. ``v_out`` (optional) receives V
    as well, e.g. the video rows of the joint attention V."""
    _ops.fused_qkv_norm_rope_cache(qkv, num_heads, eps, q_weight, k_weight, cos, sin, q_out, k_out,
                                   cache_k, cache_v, slot, slot_offset, v_out, cache_tokens, cache_pre_rope)


def fp8_qkv_norm_rope_cache(mat_a, mat_b, scales_a, scales_b, bias, num_heads, eps, q_weight, k_weight, cos, sin,
                            q_out, k_out=None, cache_k=None, cache_v=None, slot=0, slot_offset=0, v_out=None,
                            cache_tokens: int = -1, cache_pre_rope: bool = True):
    """The QKV projection (fp8_scaled_mm to bf16 [M, 3*H*D], scales as there) followed by
    fused_qkv_norm_rope_cache on its output (same arguments, cos/sin [M, D/2]), with the same
    results; the GEMM's epilogue writes the norm/RoPE/ring outputs itself where the shape allows,
    so the QKV rows are not stored in between."""
    _ops.fp8_qkv_norm_rope_cache(mat_a, mat_b, scales_a, scales_b, bias, num_heads, eps, q_weight, k_weight, cos,
                                 sin, q_out, k_out, cache_k, cache_v, slot, slot_offset, v_out, cache_tokens,
                                 cache_pre_rope)


def fused_cached_kv_pack_out(key0, value0, key1, value1, cos, sin, out_k, out_v):
    """fused_cached_kv_pack writing into caller-provided dense [1, len0 + len1, H, D] outputs,
    e.g. the cached rows at the head of the joint attention K / V."""
    _ops.fused_cached_kv_pack_out(key0, value0, key1, value1, cos, sin, out_k, out_v)


def fused_text_qkv_pack(txt_q, txt_k, txt_v, txt_q_weight, txt_k_weight, eps, out_q, out_k, out_v):
    """The condition segment of fused_joint_qkv_pack (two-rounding q/k RMSNorm, V copied) written
    into caller-provided dense [1, T, H, D] outputs (the tails of the joint Q / K / V)."""
    _ops.fused_text_qkv_pack(txt_q, txt_k, txt_v, txt_q_weight, txt_k_weight, eps, out_q, out_k, out_v)


def sdpa_attention(query, key, value, scale: Optional[float] = None):
    """softmax(q k^T * scale) v per head on [B, S, H, D] bf16 tensors, non-causal, no mask:
    the reference's ``_sdpa_attention`` (dit.py:154-167) without its transposes. scale defaults
    to 1/sqrt(D) like F.scaled_dot_product_attention; head_dim 128."""
    return _ops.sdpa_attention(query, key, value, scale)


def sdpa_attention_out(query, key, value, out, scale: Optional[float] = None):
    """sdpa_attention writing into ``out`` ([B, S, H, D], dense heads), e.g. rows of a
    [S, H*D] buffer that the out-projection quantiser reads."""
    _ops.sdpa_attention_out(query, key, value, out, scale)
