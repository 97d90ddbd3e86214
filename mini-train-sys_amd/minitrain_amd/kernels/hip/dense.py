"""The decoder's operators around its matrix products: RMSNorm, rotary encoding, attention and cross-entropy.

Each stands in for a chain of stock elementwise and reduction kernels
(minitrain/kernels/torch_ops.py of the reference) that reads and writes the activations several
times over, in fp32 on the way: here one launch forward and one or two backward, each operand read
once and each result written once.  The predicates say what the kernels take; the backend leaves
everything else (CPU tensors, other dtypes or layouts) to the stock operators.  The autograd nodes
are native (``csrc/host/mts_host.cpp``).
"""

import contextlib
import threading

import torch
from torch.overrides import has_torch_function

from minitrain_amd import _lib


def _may_replace(*tensors) -> bool:
    """The stock operators stay where a compiler traces them or a subclass wants to see them."""
    return not torch.compiler.is_compiling() and not has_torch_function(tensors)


def is_rmsnorm_supported(x, weight, residual=None) -> bool:
    return _may_replace(x, weight, residual) and _lib.host().rmsnorm_supported(x, weight, residual)


def rmsnorm(x, weight, eps: float):
    return _lib.host().rmsnorm(x, weight, eps)


def add_rmsnorm(x, residual, weight, eps: float):
    """``(x + residual, rmsnorm(x + residual))``"""
    return _lib.host().add_rmsnorm(x, residual, weight, eps)


def is_rope_supported(q, k, cos, sin) -> bool:
    return _may_replace(q, k, cos, sin) and _lib.host().rope_supported(q, k, cos, sin)


def rope(q, k, cos, sin):
    return _lib.host().rope(q, k, cos, sin)


def is_qkv_rope_supported(qkv, cos, sin, heads: int) -> bool:
    return _may_replace(qkv, cos, sin) and _lib.host().qkv_rope_supported(qkv, cos, sin, heads)


def qkv_rope(qkv, cos, sin, heads: int):
    """Rotated queries, rotated keys and values ``[B, heads, S, D]`` of the packed projection ``[B, S, 3 * heads * D]``"""
    return _lib.host().qkv_rope(qkv, cos, sin, heads)


def is_linear_supported(x, weight) -> bool:
    return _may_replace(x, weight) and _lib.host().linear_supported(x, weight)


def linear(x, weight):
    """``F.linear(x, weight)`` under autocast, with the gradient of the fp32 ``weight`` summed in fp32"""
    return _lib.host().linear(x, weight)


def is_linear_alone_supported(x, weight) -> bool:
    return _may_replace(x, weight) and _lib.host().linear_alone_supported(x, weight)


def linear_alone(x, weight):
    """``F.linear(x, weight)`` under autocast, where no gradient is wanted"""
    return _lib.host().linear_alone(x, weight)


def is_embedding_supported(ids, weight, dtype) -> bool:
    return _may_replace(ids, weight) and _lib.host().embedding_supported(ids, weight, dtype)


def embedding(ids, weight, dtype):
    """``F.embedding(ids, weight).to(dtype)`` with the gradient of ``weight`` summed from the gradient in ``dtype``"""
    return _lib.host().embedding(ids, weight, dtype)


def is_attention_supported(q, k, v) -> bool:
    return _may_replace(q, k, v) and _lib.host().attention_supported(q, k, v)


def attention(q, k, v, is_causal: bool):
    """``F.scaled_dot_product_attention(q, k, v, is_causal=is_causal)``"""
    return _lib.host().attention(q, k, v, is_causal)


def is_qkv_attention_supported(qkv, cos, sin, heads: int) -> bool:
    return _may_replace(qkv, cos, sin) and _lib.host().qkv_attention_supported(qkv, cos, sin, heads)


def qkv_attention(qkv, cos, sin, heads: int, is_causal: bool):
    """``attention(*qkv_rope(qkv, cos, sin, heads), is_causal)`` as ``[B, S, heads * D]``"""
    return _lib.host().qkv_attention(qkv, cos, sin, heads, is_causal)


def is_cross_entropy_supported(logits, targets) -> bool:
    return _may_replace(logits, targets) and _lib.host().cross_entropy_supported(logits, targets)


_root = threading.local()


@contextlib.contextmanager
def loss_is_root():
    """Losses formed inside, by this thread, are the root of the caller's backward pass, unscaled: their gradient may be formed with them."""
    before = getattr(_root, "is_loss", False)
    _root.is_loss = True
    try:
        yield
    finally:
        _root.is_loss = before


def cross_entropy(logits, targets):
    """``F.cross_entropy(logits.float(), targets)`` without the fp32 copy of the logits"""
    return _lib.host().cross_entropy(logits, targets, getattr(_root, "is_loss", False))


def is_layer_means_supported(groups, differentiable: int) -> bool:
    flat = [t for group in groups for t in group]
    return all(isinstance(t, torch.Tensor) for t in flat) and _may_replace(*flat) and _lib.host().layer_means_supported(groups, differentiable)


def layer_means(groups, differentiable: int):
    """``torch.stack(group).float().mean(0)`` of every group of tensors; gradients go to the first ``differentiable`` ones"""
    return _lib.host().layer_means(groups, differentiable)


def is_total_loss_supported(loss, aux, z) -> bool:
    return _may_replace(loss, aux, z) and _lib.host().total_loss_supported(loss, aux, z)


def total_loss(loss, aux, z, aux_coef: float, z_coef: float):
    """``loss + aux_coef * aux + z_coef * z``, and without gradients its two last terms and their sum"""
    return _lib.host().total_loss(loss, aux, z, aux_coef, z_coef)
