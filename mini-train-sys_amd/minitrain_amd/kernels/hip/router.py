"""Router post-process on the GPU: one pass over the fp32 logits.

Counterpart of minitrain/kernels/triton/router.py:262-357 (module-level entry point; the
autograd node is native, ``csrc/host/mts_host.cpp``) with the argument checks of
minitrain/kernels/torch_ops.py:96-101.  Top-k is taken on the logits with the
lower expert index winning ties, and the statistics are reduced in a fixed
order, so the operator is deterministic and needs no deterministic-mode opt-out.
"""

import torch

from minitrain_amd import _lib
from minitrain_amd.model.ops import RouterPostprocessOutput

_MAX_EXPERTS = 1024
_MAX_TOP_K = 8


def is_router_postprocess_supported(logits: torch.Tensor, top_k: int, normalize: bool) -> bool:
    del normalize  # both normalised and raw full-softmax weights are supported
    return (
        logits.is_cuda
        and logits.ndim == 2
        and logits.dtype == torch.float32
        and logits.shape[0] > 0
        and 1 <= top_k <= min(logits.shape[1], _MAX_TOP_K)
        and logits.shape[1] <= _MAX_EXPERTS
    )


def router_postprocess(logits: torch.Tensor, top_k: int, *, normalize: bool, weights_dtype=None) -> RouterPostprocessOutput:
    """Process router logits without materialising the full probability matrix.

    ``weights_dtype`` (bf16 or fp16, an extension of the reference's signature) also asks for
    ``expert_weights_cast``, the differentiable copy of the weights in that dtype."""

    if logits.ndim != 2 or logits.dtype != torch.float32:
        raise ValueError("router logits must be a 2D fp32 tensor")
    if logits.shape[0] == 0:
        raise ValueError("router logits must contain at least one token")
    if not 1 <= top_k <= logits.shape[1]:
        raise ValueError(f"top_k must be in [1, {logits.shape[1]}], got {top_k}")
    if not is_router_postprocess_supported(logits, top_k, normalize):
        raise RuntimeError(
            "hip router postprocess requires non-empty 2D fp32 logits on the GPU, "
            f"1 <= top_k <= {_MAX_TOP_K} and at most {_MAX_EXPERTS} experts"
        )
    if weights_dtype not in (None, torch.bfloat16, torch.float16):
        raise ValueError("weights_dtype must be bfloat16 or float16")
    act_dtype = -1 if weights_dtype is None else _lib.dtype_code(weights_dtype)
    weights, indices, probability_mean, z_loss, entropy, counts, load_balance, load_stats, *cast = (
        _lib.host().router_postprocess(logits, top_k, normalize, act_dtype)
    )
    return RouterPostprocessOutput(
        expert_weights=weights,
        expert_indices=indices,
        probability_per_expert=probability_mean,
        z_loss=z_loss,
        entropy=entropy,
        expert_counts=counts,
        load_balance_loss=load_balance,
        load_stats=load_stats,
        expert_weights_cast=cast[0] if cast else None,
    )


def is_router_logits_supported(hidden_states: torch.Tensor, weight: torch.Tensor) -> bool:
    return _lib.host().router_logits_supported(hidden_states, weight)


def router_logits(hidden_states: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """fp32 router logits of ``hidden_states`` [T,H] (bf16, fp16 or fp32) and ``weight`` [E,H] (fp32).

    Stands in for ``F.linear(hidden_states.float(), weight.float())`` of the reference's
    TopKRouter.forward (minitrain/model/moe_router.py:64-76).
    """

    if not is_router_logits_supported(hidden_states, weight):
        raise RuntimeError(
            "hip router_logits requires 2D bf16/fp16/fp32 activations and a 2D fp32 weight on the GPU with at most 1024 experts, "
            "and up to 16 of them a hidden size that is a multiple of 4 and at most 4096 (E * H <= 32768)"
        )
    return _lib.host().router_logits(hidden_states, weight)
