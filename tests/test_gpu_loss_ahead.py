"""Cross-entropy whose gradient is formed with the loss, because the caller says that the loss is the root of its backward pass."""

import pytest
import torch

from minitrain_amd.kernels.hip.dense import loss_is_root
from tests.helpers import hip_backend

pytestmark = pytest.mark.gpu
ULP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _loss(logits, targets, root=True):
    ops = hip_backend()
    if not root:
        return ops.cross_entropy(logits, targets)
    with loss_is_root():
        return ops.cross_entropy(logits, targets)


def _inputs(N, V, dtype):
    g = torch.Generator().manual_seed(N + V)
    logits = (4 * torch.randn(N, V, generator=g)).to(dtype)
    targets = torch.randint(0, V, (N,), generator=g)
    targets[0], targets[-1] = 0, V - 1   # the first and the last column
    if N > 3:
        targets[1] = -100
        logits[2, V // 2] = 200.0
        logits[3, :V - 1] = float("-inf")
        targets[3] = V - 1
    return logits, targets


@pytest.mark.parametrize("factor", [1.0, 3.0])
@pytest.mark.parametrize("N,V", [(1, 8), (5, 16), (4, 2048), (4, 2056), (6, 8192), (5, 8200), (5, 16384), (5, 16392), (5, 32000), (6, 32776), (4, 50256), (4, 57344), (4, 65536)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_loss_and_gradient(N, V, dtype, factor):
    """Every size of block, full and partly filled; a loss that is scaled after all."""
    print(f"loss ahead {N}x{V} {dtype} {factor}", flush=True)
    logits, targets = _inputs(N, V, dtype)
    leaf = logits.cuda().requires_grad_(True)
    loss = _loss(leaf, targets.cuda())
    grads = [torch.autograd.grad(factor * loss, leaf, retain_graph=True)[0] for _ in range(2)]   # the second is not the one formed ahead
    ref = logits.double().requires_grad_(True)
    want = torch.nn.functional.cross_entropy(ref, targets)
    (factor * want).backward()
    assert abs(loss.item() - want.item()) <= 1e-5 * max(1.0, abs(want.item()))
    for got in grads:   # differences of a probability and 1: errors are relative to 1 times the factor, also where they cancel
        bound = ULP[dtype] * factor / int((targets != -100).sum())
        assert float((got.double().cpu() - ref.grad).abs().max()) <= bound
        assert N <= 3 or not got[1].any()
    assert torch.equal(*grads) if factor != 1 else True


@pytest.mark.parametrize("N,V", [(128, 4097), (131, 50257), (256, 65535)])
@pytest.mark.parametrize("who", ["nobody", "hook", "scaled"])
def test_odd_vocabulary_behind_a_projection(N, V, who):
    """Pitched rows go to the projection, dense ones to whoever looks; the same gradients as without the word of the caller."""
    print(f"loss ahead of a projection {N}x{V} {who}", flush=True)
    g = torch.Generator().manual_seed(V)
    x0, w0 = torch.randn(N, 8, generator=g).bfloat16().cuda(), torch.randn(V, 8, generator=g).cuda()
    targets = torch.randint(0, V, (N,), generator=g).cuda()
    result = []
    for root in (True, False):
        x, w, seen = x0.clone().requires_grad_(True), w0.clone().requires_grad_(True), []
        with torch.autocast("cuda", dtype=torch.bfloat16):
            logits = hip_backend().linear(x, w)
            loss = _loss(logits, targets, root)
        if who == "hook":
            logits.register_hook(seen.append)
        (3 * loss if who == "scaled" else loss).backward()
        assert all(d.is_contiguous() for d in seen)
        result.append([loss.detach(), x.grad, w.grad, *seen])
    for a, b in zip(*result):
        assert float((a.double() - b.double()).norm()) <= 2e-3 * float(b.double().norm())   # sums in another order: a last bit of the probabilities


def test_rows_without_a_gradient_or_with_nan():
    V = 4096
    logits = torch.randn(6, V, device="cuda").bfloat16()
    logits[1, 7], logits[2, 9] = float("nan"), float("inf")
    targets = torch.tensor([3, 3, 3, V, -1, -100], device="cuda")
    grads, losses = [], []
    for root in (True, False):
        leaf = logits.clone().requires_grad_(True)
        loss = _loss(leaf, targets, root)
        loss.backward()
        losses.append(loss.detach())
        grads.append(leaf.grad)
    assert losses[0].isnan() and losses[1].isnan()
    assert torch.equal(grads[0].isnan(), grads[1].isnan()) and grads[0][1:5].isnan().all()
    assert not grads[0][5].any() and not grads[0][0].isnan().any()


def test_where_the_gradient_is_not_formed_ahead():
    """No backward pass, saved tensors that go elsewhere: the memory of the loss alone."""
    leaf = torch.randn(512, 32000, device="cuda").bfloat16().requires_grad_(True)
    targets = torch.zeros(512, dtype=torch.long, device="cuda")

    def grown(make):
        before = torch.cuda.memory_allocated()
        kept = make()
        return torch.cuda.memory_allocated() - before, kept

    size = leaf.numel() * 2
    assert grown(lambda: _loss(leaf, targets))[0] >= size
    assert grown(lambda: _loss(leaf, targets, root=False))[0] < size
    with torch.no_grad():
        assert grown(lambda: _loss(leaf, targets))[0] < size
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t):
        assert grown(lambda: _loss(leaf, targets))[0] < size
