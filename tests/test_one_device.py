"""Operands on two GPUs are not what a kernel takes: the predicates look at the device of every operand (CPU: they read sizes,
types, addresses and devices only, so host memory that is labelled as a GPU's will do)."""

import pytest
import torch

from minitrain_amd import _lib

_MEMORY = torch.zeros(4096 + 16, dtype=torch.uint8)


def _labelled(index, *shape, dtype=torch.float32):
    start = -_MEMORY.data_ptr() % 16 + _MEMORY.data_ptr()
    storage = torch._C._construct_storage_from_data_pointer(start, torch.device("cuda", index), 4096)
    stride = torch.empty(shape, device="meta").stride()
    return torch._C._construct_CUDA_Tensor_From_Storage_And_Metadata(dict(dtype=dtype, size=shape, stride=stride, storage_offset=0), storage)


def _bf16(*shape):
    return lambda index: _labelled(index, *shape, dtype=torch.bfloat16)


def _fp32(*shape):
    return lambda index: _labelled(index, *shape)


def _int(dtype, *shape):
    return lambda index: _labelled(index, *shape, dtype=dtype)


def _update_supported(h, *tensors):
    """Of tensors that are each a parameter, two moments and a step; a gradient is where its parameter is, or cannot be set."""
    for param, *_ in tensors:
        param.grad = _labelled(param.device.index, *param.shape)
    return h.adamw_supported(*map(list, zip(*tensors)))


CALLS = {
    "rmsnorm": ([_bf16(3, 8), _fp32(8)], lambda h, x, w: h.rmsnorm_supported(x, w, None)),
    "add_rmsnorm": ([_bf16(3, 8), _fp32(8), _bf16(3, 8)], lambda h, x, w, r: h.rmsnorm_supported(x, w, r)),
    "rope": ([_bf16(1, 2, 3, 4), _bf16(1, 2, 3, 4), _bf16(3, 4), _bf16(3, 4)], lambda h, *a: h.rope_supported(*a)),
    "qkv_rope": ([_bf16(1, 3, 24), _bf16(3, 4), _bf16(3, 4)], lambda h, *a: h.qkv_rope_supported(*a, 2)),
    "attention": ([_bf16(1, 1, 3, 64)] * 3, lambda h, *a: h.attention_supported(*a)),
    "cross_entropy": ([_bf16(3, 8), _int(torch.int64, 3)], lambda h, *a: h.cross_entropy_supported(*a)),
    "embedding": ([_int(torch.int64, 1, 3), _fp32(5, 8)], lambda h, ids, w: h.embedding_supported(ids, w.requires_grad_(True), torch.bfloat16)),
    "qkv_attention": ([_bf16(1, 3, 192), _bf16(3, 64), _bf16(3, 64)], lambda h, *a: h.qkv_attention_supported(*a, 1)),
    "layer_means": ([_fp32(), _fp32(), _fp32(4), _fp32(4)], lambda h, a, b, c, d: h.layer_means_supported([[a, b], [c, d]], 1)),
    "total_loss": ([_fp32()] * 3, lambda h, *a: h.total_loss_supported(*a)),
    "adamw": ([_fp32(8)] * 3 + [_fp32()] + [_fp32(4)] * 3 + [_fp32()], lambda h, *a: _update_supported(h, a[:4], a[4:])),
    "router_logits": ([_bf16(3, 8), _fp32(4, 8)], lambda h, *a: h.router_logits_supported(*a)),
    "router_logits, many experts": ([_bf16(3, 8), _fp32(20, 8)], lambda h, *a: h.router_logits_supported(*a)),
    "moe_layer": ([_bf16(3, 8), _fp32(4, 8), _bf16(4, 16, 8), _bf16(4, 8, 8)], lambda h, *a: h.layer_violation(*a, 2) is None),
    "fused_moe": ([_bf16(3, 8), _bf16(4, 16, 8), _bf16(4, 8, 8), _int(torch.int32, 3, 2), _bf16(3, 2)], lambda h, *a: h.fused_moe_violation(*a) is None),
}


@pytest.mark.parametrize("name", CALLS)
def test_operands_on_two_devices_are_refused(name):
    operands, takes = CALLS[name]
    assert takes(_lib.host(), *(make(0) for make in operands))
    for other in range(len(operands)):
        assert not takes(_lib.host(), *(make(int(i == other)) for i, make in enumerate(operands))), other
