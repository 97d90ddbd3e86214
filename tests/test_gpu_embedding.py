"""The gradient of the embedding table against fp64 sums, and which calls it is taken for."""

import pytest
import torch

from minitrain_amd.model.decoder import embed
from tests.helpers import hip_backend


def _ids(T, V, spread, g):
    if spread == "one":
        return torch.full((T,), V - 1)
    if spread == "few":   # some rows of more tokens than a wave sums alone
        return torch.randint(0, min(V, 5), (T,), generator=g) * (V // min(V, 5)) % V
    ids = torch.randint(0, V, (T,), generator=g)
    return torch.where(torch.rand(T, generator=g) < 0.5, V // 3, ids) if spread == "half" else ids


@pytest.mark.gpu
@pytest.mark.parametrize("T,V,H,spread", [(1, 1, 4, "one"), (63, 7, 256, "even"), (65, 257, 260, "even"), (1025, 1000, 768, "few"), (1000, 513, 1024, "one"),
                                          (5003, 50257, 768, "even"), (4099, 8192, 1536, "few"), (300, 33, 4096, "few"),
                                          # rows of whole segments of 128 places, alone and with others in front and behind; ranges of ids at their longest
                                          (127, 9, 512, "one"), (128, 9, 512, "one"), (8193, 3, 260, "even"), (20000, 50257, 768, "half"), (3000, 300001, 4, "even")])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_gradient_of_the_table(T, V, H, spread, dtype):
    print(f"embedding T={T} V={V} H={H} {spread} {dtype}", flush=True)
    g = torch.Generator().manual_seed(T + V)
    ids = _ids(T, V, spread, g)
    grad = torch.randn(T, H, generator=g).to(dtype)
    table = torch.nn.Embedding(V, H, device="cuda")
    out = hip_backend().embedding(ids.cuda().view(1, T), table.weight, dtype)
    assert torch.equal(out, table(ids.cuda().view(1, T)).to(dtype))
    grads = [torch.autograd.grad(out, table.weight, grad.cuda().view(1, T, H), retain_graph=True)[0] for _ in range(2)]
    assert torch.equal(*grads)   # a fixed order
    want = torch.zeros(V, H, dtype=torch.float64).index_add_(0, ids, grad.double())
    size = torch.zeros(V, H, dtype=torch.float64).index_add_(0, ids, grad.double().abs())
    most = torch.bincount(ids, minlength=V).double().clamp(min=1)[:, None]
    # n fp32 additions: each rounds a partial sum that is no larger than the sum of the magnitudes
    assert ((grads[0].double().cpu() - want).abs() <= most * 2.0 ** -24 * size).all()


@pytest.mark.gpu
def test_calls_that_stay_stock():
    ops = hip_backend()
    ids = torch.tensor([0, 3], device="cuda")
    table = torch.nn.Embedding(4, 8, device="cuda")
    assert ops.embedding(ids, table.weight, torch.bfloat16) is not None
    assert ops.embedding(ids.int(), table.weight, torch.bfloat16) is None
    assert ops.embedding(ids, table.weight.bfloat16(), torch.bfloat16) is None
    assert ops.embedding(ids.cpu(), table.weight, torch.bfloat16) is None
    with torch.no_grad():
        assert ops.embedding(ids, table.weight, torch.bfloat16) is None
    padded = torch.nn.Embedding(4, 8, padding_idx=3, device="cuda")
    embed(padded, ids, torch.bfloat16, ops).sum().backward()
    assert not padded.weight.grad[3].any() and (padded.weight.grad[0] == 1).all()
    weight = torch.randn(4, 8, device="cuda", requires_grad=True)   # a gradient that is itself differentiated
    x = ops.embedding(ids, weight, torch.float32)
    first, = torch.autograd.grad(x.square().sum(), weight, create_graph=True)
    second, = torch.autograd.grad(first.sum(), weight)
    assert (second[[0, 3]] == 2).all() and not second[[1, 2]].any()
