"""The whole MoE layer (router projection, post-process, routing metadata, experts, combine) as one
autograd node.

The reference composes the layer from three autograd nodes (minitrain/model/moe_router.py:64-90 and
minitrain/model/blocks.py:86-102): ``F.linear`` for the router logits, ``router_postprocess`` and
``fused_moe``.  The activations feed two of them, so autograd sums two gradients for ``x`` with one more
kernel, and every node boundary is a launch boundary.  Here the forward pass starts with the chained
head (two launches: projection + post-process, then scatter + statistics; one for few tokens) and the backward pass
forms the router's gradient before the dX combine, which adds it to the experts' gradient in the same
pass.  Same arithmetic as the separate operators; it is an extension the MoE block uses when the backend
offers it (``ops.moe_layer``) and the configuration allows it.
"""

import torch

from minitrain_amd import _lib
from minitrain_amd.kernels.hip.fused_moe import dw_workspace_limit
from minitrain_amd.kernels.hip.switches import SWITCHES


def moe_layer_violation(x, router_weight, gate_up_proj, down_proj, top_k: int):
    """The first requirement of the layer contract that the arguments miss, or None."""
    if not all(isinstance(t, torch.Tensor) for t in (x, router_weight, gate_up_proj, down_proj)):
        return "x, router_weight, gate_up_proj and down_proj are tensors"
    return _lib.host().layer_violation(x, router_weight, gate_up_proj, down_proj, top_k)


def moe_layer(x, router_weight, gate_up_proj, down_proj, top_k: int, *, normalize: bool, capacity: int | None = None):
    """``(hidden, load_balance_loss, z_loss, probability_per_expert, entropy, expert_counts, load_stats,
    expert_indices, expert_weights)`` of one MoE layer on ``x [T,H]``; the first four are differentiable.
    With ``capacity`` an expert accepts its that many most confident routes (the rule of ``capacity_mask``): the others get
    no row, a token's kept weights are renormalised with ``normalize``, and ``load_stats`` describes the accepted routes;
    ``expert_counts``, ``expert_indices`` and ``expert_weights`` stay those of the unlimited routing.
    The autograd node is native (``csrc/host/mts_host.cpp``)."""
    missed = moe_layer_violation(x, router_weight, gate_up_proj, down_proj, top_k)
    if missed is not None:
        raise RuntimeError(f"Unsupported tensor contract for the hip MoE layer: it requires {missed}")
    return run_moe_layer(x, router_weight, gate_up_proj, down_proj, top_k, normalize, capacity)


def run_moe_layer(x, router_weight, gate_up_proj, down_proj, top_k: int, normalize: bool, capacity: int | None):
    """:func:`moe_layer` for arguments that are known to fit the contract."""
    return _lib.host().moe_layer(x, router_weight, gate_up_proj, down_proj, top_k, normalize, -1 if capacity is None else capacity,
                                 SWITCHES.mask(), dw_workspace_limit(x, gate_up_proj))
