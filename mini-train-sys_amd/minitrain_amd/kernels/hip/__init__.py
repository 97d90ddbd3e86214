"""`hip` operator backend: MoE operators on hand-written gfx950 kernels.

Counterpart of the reference's ``TritonOpsBackend``
(minitrain/kernels/triton/__init__.py:36-113) for the two MoE methods.  Unlike
that class there is no fallback: an unsupported tensor contract raises.
"""

import torch.nn.functional as F

from minitrain_amd.kernels.dense_ops import DenseTorchOps
from minitrain_amd.kernels.hip import dense
from minitrain_amd.kernels.hip.capacity import capacity_mask, is_capacity_mask_supported
from minitrain_amd.kernels.hip.fused_moe import expert_counts, fused_moe, is_fused_moe_supported
from minitrain_amd.kernels.hip.moe_layer import moe_layer, moe_layer_violation, run_moe_layer
from minitrain_amd.kernels.hip.switches import SWITCHES
from minitrain_amd.kernels.hip.router import (
    is_router_logits_supported,
    is_router_postprocess_supported,
    router_logits,
    router_postprocess,
)


class HipOpsBackend(DenseTorchOps):
    name = "hip"
    # fused_moe gives a route whose expert index is negative no row in the expert GEMMs
    drops_routes = True

    # router_postprocess takes ``weights_dtype`` and then also returns the weights rounded to it
    # (a comparison switch leaves the cast to the caller, see switches.py)
    casts_router_weights = SWITCHES.router_cast

    def router_postprocess(self, logits, top_k, *, normalize, weights_dtype=None):
        return router_postprocess(logits, top_k, normalize=normalize, weights_dtype=weights_dtype)

    def fused_moe(self, x, gate_up_proj, down_proj, top_k_index, top_k_weights):
        return fused_moe(x, gate_up_proj, down_proj, top_k_index, top_k_weights)

    # The decoder's operators around its matrix products: one kernel where the stock operators are a chain of
    # elementwise and reduction kernels; what the kernels do not take (CPU tensors, other types and layouts) stays stock.

    def _are_own(self, names) -> bool:
        """Whether these operators are this class's, so that a fused form may stand in for them."""
        cls, instance = type(self), self.__dict__
        for name in names:
            if name in instance or getattr(cls, name) is not _OWN[name]:
                return False
        return True

    def rmsnorm(self, x, weight, eps):
        if dense.is_rmsnorm_supported(x, weight):
            return dense.rmsnorm(x, weight, eps)
        return super().rmsnorm(x, weight, eps)

    def add_rmsnorm(self, x, residual, weight, eps):
        """Extension: ``(x + residual, rmsnorm(x + residual))`` in one pass."""
        if self._are_own(("rmsnorm",)) and dense.is_rmsnorm_supported(x, weight, residual):
            return dense.add_rmsnorm(x, residual, weight, eps)
        total = x + residual
        return total, self.rmsnorm(total, weight, eps)

    def rope(self, q, k, cos, sin):
        if dense.is_rope_supported(q, k, cos, sin):
            return dense.rope(q, k, cos, sin)
        return super().rope(q, k, cos, sin)

    def qkv_rope(self, qkv, cos, sin, heads):
        """Extension: rotated queries and keys and the values ``[B, heads, S, D]`` of a packed projection, or None when
        the kernel does not take it (the caller then splits the projection and calls ``rope``)."""
        if not self._are_own(("rope",)) or not dense.is_qkv_rope_supported(qkv, cos, sin, heads):
            return None
        return dense.qkv_rope(qkv, cos, sin, heads)

    def linear(self, x, weight):
        """Extension: ``F.linear(x, weight)``, or None where the caller's own does as well."""
        if dense.is_linear_supported(x, weight):
            return dense.linear(x, weight)
        if dense.is_linear_alone_supported(x, weight):
            return dense.linear_alone(x, weight)
        return None

    def embedding(self, ids, weight, dtype):
        """Extension: ``F.embedding(ids, weight).to(dtype)`` whose gradient is this backend's, or None where the caller's own does as well."""
        if not dense.is_embedding_supported(ids, weight, dtype):
            return None
        return dense.embedding(ids, weight, dtype)

    def attention(self, q, k, v, *, is_causal, dropout_p):
        if not dropout_p and dense.is_attention_supported(q, k, v):
            return dense.attention(q, k, v, is_causal)
        return super().attention(q, k, v, is_causal=is_causal, dropout_p=dropout_p)

    def qkv_attention(self, qkv, cos, sin, heads, *, is_causal, dropout_p):
        """Extension: ``attention`` of what ``qkv_rope`` returns, as ``[B, S, heads * D]``, or None when the kernels do not take it or one of
        the operators that it stands for is overridden."""
        if dropout_p or not self._are_own(("rope", "qkv_rope", "attention")) or not dense.is_qkv_attention_supported(qkv, cos, sin, heads):
            return None
        return dense.qkv_attention(qkv, cos, sin, heads, is_causal)

    def cross_entropy(self, logits, targets):
        if dense.is_cross_entropy_supported(logits, targets):
            return dense.cross_entropy(logits, targets)
        return super().cross_entropy(logits, targets)

    def fused_linear_cross_entropy(self, x, weight, targets):
        logits = self.linear(x, weight)
        return self.cross_entropy(F.linear(x, weight) if logits is None else logits, targets)

    def layer_means(self, groups, differentiable):
        """Extension: the mean over the layers of every group of tensors in one launch (the first ``differentiable`` groups
        are single numbers that carry gradients), or None when the kernel does not take them."""
        if not dense.is_layer_means_supported(groups, differentiable):
            return None
        return dense.layer_means(groups, differentiable)

    def total_loss(self, loss, aux, z, aux_coef, z_coef):
        """Extension: ``(loss + aux_coef * aux + z_coef * z, aux_coef * aux, z_coef * z, their sum)``, the last three without
        gradients, or None when the kernel does not take them."""
        if not (isinstance(aux_coef, (int, float)) and isinstance(z_coef, (int, float)) and dense.is_total_loss_supported(loss, aux, z)):
            return None
        return dense.total_loss(loss, aux, z, aux_coef, z_coef)

    def expert_counts(self, expert_indices, num_experts):
        """Extension: routes per expert (int32 ``[E]``) without a host synchronisation."""
        return expert_counts(expert_indices, num_experts)

    def capacity_mask(self, expert_indices, expert_weights, num_experts, capacity):
        """Extension: ``(keep, kept_index, accepted)`` of a capacity-limited dispatch, or None when
        the contract is not supported (the caller then uses its own sort-based selection)."""
        if not is_capacity_mask_supported(expert_indices, expert_weights, num_experts):
            return None
        return capacity_mask(expert_indices, expert_weights, num_experts, capacity)

    # a comparison switch keeps the layer on the three separate operators (switches.py); an instance may also set
    # this attribute to False (the one-node path does not call the router module; the block does not take it when that
    # module has hooks or a forward of its own)
    offers_moe_layer = SWITCHES.layer_node

    # moe_layer takes a capacity limit
    limits_moe_layer = True

    def moe_layer(self, x, router_weight, gate_up_proj, down_proj, top_k, *, normalize, capacity=None):
        """Extension: router projection, post-process, routing metadata and the experts as one autograd
        node (see ``kernels/hip/moe_layer.py``).  Returns None when the contract is not supported or one of the
        operators that it stands for is overridden; the caller then composes the layer from them."""
        operators = _OF_LAYER if capacity is None else _OF_LIMITED_LAYER
        if not self.offers_moe_layer or not self._are_own(operators) or moe_layer_violation(x, router_weight, gate_up_proj, down_proj, top_k) is not None:
            return None
        return run_moe_layer(x, router_weight, gate_up_proj, down_proj, top_k, normalize, capacity)

    def router_logits(self, hidden_states, weight):
        """Extension beyond the reference's operator interface: the router projection in fp32
        straight from the activation dtype.  Returns None when the contract is not supported,
        and the caller then runs its own ``F.linear``."""
        if not is_router_logits_supported(hidden_states, weight):
            return None
        return router_logits(hidden_states, weight)


_OF_LAYER = ("router_logits", "router_postprocess", "fused_moe")
_OF_LIMITED_LAYER = (*_OF_LAYER, "capacity_mask")
_OWN = {name: getattr(HipOpsBackend, name) for name in ("rmsnorm", "rope", "qkv_rope", "attention", *_OF_LIMITED_LAYER)}

__all__ = [
    "HipOpsBackend",
    "capacity_mask",
    "expert_counts",
    "fused_moe",
    "is_capacity_mask_supported",
    "is_fused_moe_supported",
    "is_router_logits_supported",
    "is_router_postprocess_supported",
    "moe_layer",
    "router_logits",
    "router_postprocess",
]
