"""Modules that do not run their class's own forward are called, not replaced by a fused form of it (CPU)."""

import pytest
import torch
from torch import nn

from minitrain_amd.kernels.dense_ops import DenseTorchOps
from minitrain_amd.model.blocks import FeedForwardOutput, MoEFeedForward
from minitrain_amd.model.config import ModelConfig
from minitrain_amd.model.decoder import MiniTransformer, RMSNorm


class FusedOps(DenseTorchOps):
    def add_rmsnorm(self, x, residual, weight, eps):
        return x + residual, self.rmsnorm(x + residual, weight, eps)


class HalfFeedForward(nn.Module):
    def forward(self, x, ops):
        return FeedForwardOutput(hidden_states=0.5 * x, router_aux_loss=x.new_zeros(()), router_z_loss=x.new_zeros(()))


class Wrapper(nn.Module):
    """As data-parallel and checkpointing wrappers do: attributes of the module inside, a forward of its own."""

    def __init__(self, module, calls):
        super().__init__()
        self.module, self.calls = module, calls

    def __getattr__(self, name):
        try:
            return super().__getattr__(name)
        except AttributeError:
            return getattr(super().__getattr__("module"), name)

    def forward(self, *args):
        self.calls.append(1)
        return self.module(*args)


def _wrap_block(model, calls):
    model.blocks[1] = Wrapper(model.blocks[1], calls)


def _own_forward(model, calls):
    block = model.blocks[0]
    inner = block.forward
    block.forward = lambda *a: (calls.append(1), inner(*a))[1]


def _hooked_block(model, calls):
    model.blocks[0].register_forward_hook(lambda *a: calls.append(1))


def _hooked_norm(model, calls):
    model.blocks[1].attn_norm.register_forward_pre_hook(lambda *a: calls.append(1))


def _wrap_norm(model, calls):
    model.norm = Wrapper(model.norm, calls)


def _norm_subclass(model, calls):
    class Counted(RMSNorm):
        def forward(self, x, ops):
            calls.append(1)
            return super().forward(x, ops)

    model.blocks[0].ffn_norm.__class__ = Counted


@pytest.mark.parametrize("change", [_wrap_block, _own_forward, _hooked_block, _hooked_norm, _wrap_norm, _norm_subclass])
def test_changed_modules_are_called(change):
    torch.manual_seed(0)
    cfg = ModelConfig(vocab_size=50, seq_len=8, n_layers=2, n_heads=2, hidden_size=16, intermediate_size=32, num_experts=4, experts_per_token=2)
    model = MiniTransformer(cfg, FusedOps())
    for block in model.blocks:
        block.ffn = HalfFeedForward()
    ids = torch.randint(0, 50, (2, 8))
    plain = model(ids)[1]
    calls = []
    change(model, calls)
    assert torch.equal(model(ids)[1], plain)
    assert calls == [1]


def test_hooked_router_is_called():
    """The layer as one node does not call the router module: with a hook on it the block composes the layer."""
    cfg = ModelConfig(hidden_size=16, n_heads=1, intermediate_size=32, num_experts=4, experts_per_token=2, expert_capacity_factor=1.0)
    block = MoEFeedForward(cfg)

    class Ops:
        limits_moe_layer = True

        def moe_layer(self, *args, **kwargs):
            raise AssertionError("the router module is left out")

    block.router.register_forward_hook(lambda *a: None)
    assert block._whole_layer(torch.randn(4, 16), Ops()) is None
