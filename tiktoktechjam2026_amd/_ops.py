"""``torch.library`` custom operators over the C ABI (``include/mpk.h``).

Each operator is opaque to ``torch.compile``: Dynamo records it as one node,
Inductor calls it as an external kernel, and the fake (meta) implementation
gives the output shapes and dtypes without touching the device.  That is what
lets the reference CLI's default ``torch.compile(model, mode="reduce-overhead")``
(``mixed_precision_benchmark.py:86-90`` -> ``torch_transformer_benchmark.py:800-805``)
trace the module's forward in one graph and capture it in a HIP graph.

The GPU kernels are native (``csrc/torch_ops.cpp`` -> ``libmpk_ops.so``, registered
for the CUDA dispatch key when it is loaded): they check 16-byte alignment
(``ValueError``), allocate the outputs on the input's device and launch on torch's
current stream.  The Python bodies below run only until the first call has loaded that
library; there is no other implementation.
Shape, dtype and layout validation stays in the public wrappers
(``mixed_precision/hip_linear.py``, ``hip_fused.py``,
``custom_kernel/hip_attention.py``), which raise the reference's
``ValueError`` messages before any operator is called.

dtype arguments are the C ABI codes: 0 = FP32, 1 = FP16.
"""


from typing import List, Optional, Tuple

import torch

from . import _lib

_DTYPES = {_lib.F32: torch.float32, _lib.F16: torch.float16}


def _dtype(code: int) -> torch.dtype:
    try:
        return _DTYPES[int(code)]
    except KeyError:
        raise ValueError(f"unknown dtype code {code}") from None


def _native(op: str, gpu: torch.Tensor, *args):
    """Load the native kernels and run ``op`` on them (they take precedence over the Python
    bodies for GPU tensors from then on)."""
    if not gpu.is_cuda:
        raise ValueError(f"mpk::{op} requires GPU tensors")
    _lib.load_ops()
    return getattr(torch.ops.mpk, op).default(gpu, *args)


# --------------------------------------------------------------------------- LayerNorm


@torch.library.custom_op("mpk::layer_norm", mutates_args=())
def layer_norm(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor, eps: float, out_dtype: int) -> torch.Tensor:
    """``LayerNorm(x)`` of an FP32 stream with FP32 statistics (``mpk_layernorm``, no update)."""
    return _native("layer_norm", x, weight, bias, eps, out_dtype)


@layer_norm.register_fake
def _(x, weight, bias, eps, out_dtype):
    return x.new_empty(x.shape, dtype=_dtype(out_dtype))


@torch.library.custom_op("mpk::add_layer_norm", mutates_args=())
def add_layer_norm(
    x: torch.Tensor, update: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor, eps: float, out_dtype: int
) -> Tuple[torch.Tensor, torch.Tensor]:
    """``r = x + update`` (FP32) and ``LayerNorm(r)`` (``mpk_layernorm``)."""
    return _native("add_layer_norm", x, update, weight, bias, eps, out_dtype)


@add_layer_norm.register_fake
def _(x, update, weight, bias, eps, out_dtype):
    return torch.empty_like(x), x.new_empty(x.shape, dtype=_dtype(out_dtype))


# --------------------------------------------------------------------------- projections


@torch.library.custom_op("mpk::linear", mutates_args=())
def linear(
    x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor, out_dtype: int, gelu: bool, variant: int
) -> torch.Tensor:
    """``act(fp16(x) W^T + b)`` (``mpk_linear``)."""
    return _native("linear", x, weight, bias, out_dtype, gelu, variant)


@linear.register_fake
def _(x, weight, bias, out_dtype, gelu, variant):
    return x.new_empty((*x.shape[:-1], weight.shape[0]), dtype=_dtype(out_dtype))


@torch.library.custom_op("mpk::linear_qscaled", mutates_args=())
def linear_qscaled(
    x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor, out_dtype: int, q_cols: int, q_scale: float,
    variant: int,
) -> torch.Tensor:
    """``fp16(x) W^T + b`` with columns below ``q_cols`` multiplied by ``q_scale`` before the
    output rounding (``mpk_linear_qscaled``)."""
    return _native("linear_qscaled", x, weight, bias, out_dtype, q_cols, q_scale, variant)


@linear_qscaled.register_fake
def _(x, weight, bias, out_dtype, q_cols, q_scale, variant):
    return x.new_empty((*x.shape[:-1], weight.shape[0]), dtype=_dtype(out_dtype))


@torch.library.custom_op("mpk::linear_residual", mutates_args=())
def linear_residual(
    x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor, residual: torch.Tensor, variant: int
) -> torch.Tensor:
    """``fp16(x) W^T + b + residual`` in FP32 (``mpk_linear_residual``)."""
    return _native("linear_residual", x, weight, bias, residual, variant)


@linear_residual.register_fake
def _(x, weight, bias, residual, variant):
    return torch.empty_like(residual)


@torch.library.custom_op("mpk::linear_residual_into", mutates_args=("out",))
def linear_residual_into(
    x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor, residual: torch.Tensor, out: torch.Tensor, variant: int
) -> None:
    """As ``linear_residual`` into a caller-supplied FP32 ``out`` (which may be ``residual``)."""
    _native("linear_residual_into", x, weight, bias, residual, out, variant)


@linear_residual_into.register_fake
def _(x, weight, bias, residual, out, variant):
    return None


@torch.library.custom_op("mpk::linear_residual_layer_norm", mutates_args=())
def linear_residual_layer_norm(
    x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor, residual: torch.Tensor, gamma: torch.Tensor,
    beta: torch.Tensor, eps: float, out_dtype: int, variant: int,
) -> Tuple[torch.Tensor, torch.Tensor]:
    """Square projection + residual + LayerNorm with whole rows per wave (``mpk_linear_residual_layernorm``)."""
    return _native("linear_residual_layer_norm", x, weight, bias, residual, gamma, beta, eps, out_dtype, variant)


@linear_residual_layer_norm.register_fake
def _(x, weight, bias, residual, gamma, beta, eps, out_dtype, variant):
    return torch.empty_like(residual), residual.new_empty(residual.shape, dtype=_dtype(out_dtype))


@torch.library.custom_op("mpk::linear_add_layer_norm", mutates_args=())
def linear_add_layer_norm(
    x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor, residual: torch.Tensor, gamma: torch.Tensor,
    beta: torch.Tensor, eps: float, out_dtype: int,
) -> Tuple[torch.Tensor, torch.Tensor]:
    """Projection (any input width) + residual + LayerNorm on large GEMM tiles (``mpk_linear_add_layernorm``)."""
    return _native("linear_add_layer_norm", x, weight, bias, residual, gamma, beta, eps, out_dtype)


@linear_add_layer_norm.register_fake
def _(x, weight, bias, residual, gamma, beta, eps, out_dtype):
    return torch.empty_like(residual), residual.new_empty(residual.shape, dtype=_dtype(out_dtype))


@torch.library.custom_op("mpk::ffn_residual_layer_norm", mutates_args=())
def ffn_residual_layer_norm(
    x: torch.Tensor, w_in: torch.Tensor, b_in: torch.Tensor, w_out: torch.Tensor, b_out: torch.Tensor,
    residual: torch.Tensor, gamma: torch.Tensor, beta: torch.Tensor, eps: float, out_dtype: int, variant: int,
) -> Tuple[torch.Tensor, torch.Tensor]:
    """Whole FFN (hidden on chip) + residual + LayerNorm (``mpk_ffn_residual_layernorm``)."""
    return _native("ffn_residual_layer_norm", x, w_in, b_in, w_out, b_out, residual, gamma, beta, eps, out_dtype,
                   variant)


@ffn_residual_layer_norm.register_fake
def _(x, w_in, b_in, w_out, b_out, residual, gamma, beta, eps, out_dtype, variant):
    return torch.empty_like(residual), residual.new_empty(residual.shape, dtype=_dtype(out_dtype))


@torch.library.custom_op("mpk::ffn_residual_layer_norm_into", mutates_args=("normalized",))
def ffn_residual_layer_norm_into(
    x: torch.Tensor, w_in: torch.Tensor, b_in: torch.Tensor, w_out: torch.Tensor, b_out: torch.Tensor,
    residual: torch.Tensor, gamma: torch.Tensor, beta: torch.Tensor, eps: float, variant: int,
    normalized: torch.Tensor, store_residual: bool,
) -> torch.Tensor:
    """``ffn_residual_layer_norm`` with the normalized output written into ``normalized``
    (contiguous, residual's shape, FP32 or FP16: a caller's preallocated output slice, so
    no copy follows); returns the residual output, or an empty tensor when
    ``store_residual`` is false (the kernel then stores only the normalized output)."""
    return _native("ffn_residual_layer_norm_into", x, w_in, b_in, w_out, b_out, residual, gamma, beta, eps,
                   variant, normalized, store_residual)


@ffn_residual_layer_norm_into.register_fake
def _(x, w_in, b_in, w_out, b_out, residual, gamma, beta, eps, variant, normalized, store_residual):
    return torch.empty_like(residual) if store_residual else residual.new_empty(0)


@torch.library.custom_op("mpk::ffn_residual_layer_norm_final", mutates_args=())
def ffn_residual_layer_norm_final(
    x: torch.Tensor, w_in: torch.Tensor, b_in: torch.Tensor, w_out: torch.Tensor, b_out: torch.Tensor,
    residual: torch.Tensor, gamma: torch.Tensor, beta: torch.Tensor, eps: float, out_dtype: int, variant: int,
) -> torch.Tensor:
    """``ffn_residual_layer_norm`` for a last layer: only the normalized output is stored and
    returned (the residual stream after it is not read)."""
    return _native("ffn_residual_layer_norm_final", x, w_in, b_in, w_out, b_out, residual, gamma, beta, eps,
                   out_dtype, variant)


@ffn_residual_layer_norm_final.register_fake
def _(x, w_in, b_in, w_out, b_out, residual, gamma, beta, eps, out_dtype, variant):
    return residual.new_empty(residual.shape, dtype=_dtype(out_dtype))


# --------------------------------------------------------------------------- attention


@torch.library.custom_op("mpk::attention", mutates_args=())
def attention(
    q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, key_valid: Optional[torch.Tensor], scale: float, causal: bool,
    out_dtype: int, variant: int,
) -> torch.Tensor:
    """Flash attention over strided ``[B, H, S, hd]`` views -> contiguous ``[B, S, H, hd]``
    (``mpk_causal_attention``).  ``key_valid``: optional uint8 ``[B, S]``, nonzero = valid key."""
    return _native("attention", q, k, v, key_valid, scale, causal, out_dtype, variant)


@attention.register_fake
def _(q, k, v, key_valid, scale, causal, out_dtype, variant):
    batch, heads, seq_len, head_dim = q.shape
    return q.new_empty((batch, seq_len, heads, head_dim), dtype=_dtype(out_dtype))


@torch.library.custom_op("mpk::attention_prescaled", mutates_args=())
def attention_prescaled(
    q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, key_valid: Optional[torch.Tensor], causal: bool,
    out_dtype: int, variant: int,
) -> torch.Tensor:
    """Flash attention over FP16 views whose q already holds q * scale * log2(e)
    (``mpk_causal_attention_prescaled``) -> contiguous ``[B, S, H, hd]``."""
    return _native("attention_prescaled", q, k, v, key_valid, causal, out_dtype, variant)


@attention_prescaled.register_fake
def _(q, k, v, key_valid, causal, out_dtype, variant):
    batch, heads, seq_len, head_dim = q.shape
    return q.new_empty((batch, seq_len, heads, head_dim), dtype=_dtype(out_dtype))


# --------------------------------------------------------------------------- whole-layer fusions


@torch.library.custom_op("mpk::layer_norm_qkv", mutates_args=())
def layer_norm_qkv(
    x: torch.Tensor, ln_w: torch.Tensor, ln_b: torch.Tensor, w_qkv: torch.Tensor, b_qkv: torch.Tensor, eps: float,
    variant: int, q_scale: float = 0.0,
) -> torch.Tensor:
    """``fp16(LayerNorm(x)) W_qkv^T + b`` -> FP16 ``[..., 3D]`` (``mpk_layernorm_qkv``); with
    ``q_scale`` != 0 the q columns are multiplied by it before the FP16 rounding
    (``mpk_layernorm_qkv_qscaled``)."""
    return _native("layer_norm_qkv", x, ln_w, ln_b, w_qkv, b_qkv, eps, variant, q_scale)


@layer_norm_qkv.register_fake
def _(x, ln_w, ln_b, w_qkv, b_qkv, eps, variant, q_scale=0.0):
    return x.new_empty((*x.shape[:-1], 3 * x.shape[-1]), dtype=torch.float16)


@torch.library.custom_op("mpk::layer_tail", mutates_args=())
def layer_tail(
    ctx: torch.Tensor, residual: torch.Tensor, tensors: List[torch.Tensor], w_qkv: Optional[torch.Tensor],
    b_qkv: Optional[torch.Tensor], ln2_eps: float, next_eps: float, variant: int, q_scale: float = 0.0,
) -> Tuple[torch.Tensor, torch.Tensor]:
    """Out-projection through the next layer's QKV (or the final LayerNorm) in one kernel (``mpk_layer_tail``).

    ``tensors`` = [w_o, b_o, ln2_w, ln2_b, w_in, b_in, w_out, b_out, next_ln_w, next_ln_b].
    Returns ``(residual_out, qkv FP16 [..., 3D])``, or ``(residual_out, normalized FP32)``
    when ``w_qkv`` is None (last layer).  ``q_scale`` != 0 multiplies the next q columns by it
    before the FP16 rounding (``mpk_layer_tail_qscaled``).
    """
    return _native("layer_tail", ctx, residual, tensors, w_qkv, b_qkv, ln2_eps, next_eps, variant, q_scale)


@layer_tail.register_fake
def _(ctx, residual, tensors, w_qkv, b_qkv, ln2_eps, next_eps, variant, q_scale=0.0):
    d = ctx.shape[-1]
    if w_qkv is None:
        return torch.empty_like(residual), ctx.new_empty(ctx.shape, dtype=torch.float32)
    return torch.empty_like(residual), ctx.new_empty((*ctx.shape[:-1], 3 * d), dtype=torch.float16)


@torch.library.custom_op("mpk::attention_layer_tail", mutates_args=())
def attention_layer_tail(
    qkv: torch.Tensor, residual: torch.Tensor, tensors: List[torch.Tensor], w_qkv: Optional[torch.Tensor],
    b_qkv: Optional[torch.Tensor], heads: int, scale: float, causal: bool, ln2_eps: float, next_eps: float,
) -> Tuple[torch.Tensor, torch.Tensor]:
    """Attention (head dim 32) from this layer's packed ``qkv [B, S, 3D]`` through the next
    layer's QKV (or the final LayerNorm) in one kernel (``mpk_attention_layer_tail``).

    ``tensors`` as for ``layer_tail``.  Returns ``(residual_out, next qkv FP16 [B, S, 3D])``,
    or ``(residual_out, normalized FP32)`` when ``w_qkv`` is None (last layer); the next
    layer's QKV is always a new tensor (the kernel reads ``qkv`` while it writes it).
    """
    return _native("attention_layer_tail", qkv, residual, tensors, w_qkv, b_qkv, heads, scale, causal, ln2_eps,
                   next_eps)


@attention_layer_tail.register_fake
def _(qkv, residual, tensors, w_qkv, b_qkv, heads, scale, causal, ln2_eps, next_eps):
    d = residual.shape[-1]
    if w_qkv is None:
        return torch.empty_like(residual), residual.new_empty(residual.shape, dtype=torch.float32)
    return torch.empty_like(residual), residual.new_empty((*residual.shape[:-1], 3 * d), dtype=torch.float16)
