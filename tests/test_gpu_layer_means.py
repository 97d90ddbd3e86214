"""Means over the layers and the sum of the losses, against the stock operators."""

import pytest
import torch

from tests.helpers import hip_backend

pytestmark = pytest.mark.gpu


def _groups(layers, experts, seed=0):
    g = torch.Generator().manual_seed(seed)
    numbers = lambda: [torch.randn((), generator=g).cuda() for _ in range(layers)]
    vectors = [torch.randn(experts, generator=g).cuda() for _ in range(layers)]
    counts = [torch.randint(0, 9, (), generator=g).cuda() for _ in range(layers)]
    return [numbers(), numbers()], [numbers(), vectors, counts, [v[1:] for v in vectors] if experts > 1 else numbers()]


# 64 threads a group; at most 16 groups and 384 tensors a launch
@pytest.mark.parametrize("layers,experts", [(1, 1), (2, 63), (3, 64), (12, 65), (64, 1024)])
def test_means_equal_stock(layers, experts):
    ops = hip_backend()
    losses, records = _groups(layers, experts)
    got = ops.layer_means([*losses, *records], 2)
    assert got is not None
    for values, mean in zip([*losses, *records], got):
        want = torch.stack(values).double().mean(0)
        assert mean.dtype == torch.float32 and mean.shape == want.shape
        # sums of `layers` values of order one in fp32
        torch.testing.assert_close(mean.double(), want, rtol=0, atol=layers * 4 * 2**-24 * 9)


def test_loss_and_its_gradients_equal_stock():
    ops = hip_backend()
    results = []
    for fused in (True, False):
        losses, records = _groups(12, 8)
        leaves = [t.requires_grad_(True) for group in losses for t in group]
        lm = torch.tensor(3.25, device="cuda", requires_grad=True)
        if fused:
            aux, z, *_ = ops.layer_means([*losses, *records], 2)
            total, wa, wz, reg = ops.total_loss(lm, aux, z, 0.01, 0.001)
            assert not (wa.requires_grad or wz.requires_grad or reg.requires_grad)
        else:
            aux, z = (torch.stack(g).mean() for g in losses)
            wa, wz = 0.01 * aux, 0.001 * z
            total, reg = lm + wa + wz, wa + wz
        (total * 2).backward()
        results.append([total, wa, wz, reg, lm.grad, *[t.grad for t in leaves]])
    for a, b in zip(*results):
        torch.testing.assert_close(a.detach(), b.detach(), rtol=4e-7, atol=1e-9)   # a few roundings of the mean


def test_infinite_parts_stay_visible():
    ops = hip_backend()
    one, inf = torch.ones((), device="cuda"), torch.full((), float("inf"), device="cuda")
    assert torch.isnan(ops.total_loss(one, inf, one, 0.0, 0.001)[0])   # 0 * inf, as the stock operators have it


def test_what_the_kernels_do_not_take():
    ops = hip_backend()
    losses, records = _groups(2, 4)
    assert ops.layer_means([*losses, *_groups(200, 4)[1]], 2) is None                            # too many tensors
    assert ops.layer_means([*losses, [t.double() for t in records[0]]], 2) is None
    assert ops.layer_means([*losses, [t.cpu() for t in records[0]]], 2) is None
    assert ops.layer_means([*losses, [t.clone().requires_grad_(True) for t in records[0]]], 2) is None   # records carry no gradient
    assert ops.layer_means([*losses, [records[1][0], records[1][0][:2]]], 2) is None             # of different sizes
    assert ops.total_loss(losses[0][0].double(), losses[0][1], losses[1][0], 1.0, 1.0) is None


def test_coefficients_that_are_tensors_keep_their_gradients():
    """A coefficient may be learned or changed in place: the stock operators, on the GPU, with its gradient."""
    from minitrain_amd.model.decoder import total_loss

    loss, aux, z = (torch.full((), v, device="cuda") for v in (3.0, 2.0, 0.5))
    a = torch.tensor(0.25, device="cuda", requires_grad=True)
    total, weighted, *_ = total_loss(loss, aux, z, a, 2, hip_backend())
    total.backward()
    assert float(total) == 4.5 and float(weighted) == 0.5 and float(a.grad) == 2.0
