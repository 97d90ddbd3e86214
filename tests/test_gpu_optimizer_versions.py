"""What the optimizer update writes besides parameters and state, and what it marks as written, against stock clipping and fused AdamW."""

import pytest
import torch

from tests.test_gpu_optimizer import Bag, _optimizer

pytestmark = pytest.mark.gpu


def _step(bag, opt, limit, own):
    """A second step (the first makes the state), with graphs that have saved a gradient and a parameter: whether they notice."""
    from minitrain_amd.train.update import plan

    for p, g in zip(bag.p, bag.grads):
        p.grad = g.clone()
    opt.step()
    for p, g in zip(bag.p, bag.grads):
        p.grad = g.clone()
    x = torch.ones_like(bag.p[0], requires_grad=True)
    of_gradient, of_parameter = (x * bag.p[0].grad).sum(), (x * bag.p[0].detach()).sum()
    loss = torch.ones((), device="cuda")
    if own:
        update = plan(bag, opt, loss, limit)
        update.apply(update.norm(limit, loss), True)
    else:
        if limit is not None:
            torch.nn.utils.clip_grad_norm_(bag.parameters(), limit)
        opt.step()
    noticed = []
    for result in (of_gradient, of_parameter):
        try:
            result.backward()
            noticed.append(False)
        except RuntimeError as e:
            assert "modified by an inplace operation" in str(e)
            noticed.append(True)
    return noticed


@pytest.mark.parametrize("limit", [None, 1e-3, 1e9])
def test_a_graph_that_saved_a_gradient_notices_the_clipping(limit):
    runs = []
    for own in (True, False):
        bag = Bag([5, 4097])
        runs.append(_step(bag, _optimizer(bag), limit, own))
    assert runs[0][0] == runs[1][0] == (limit is not None)


@pytest.mark.parametrize("limit", [None, 1e-3])
def test_a_graph_that_saved_a_parameter_goes_on_as_after_a_stock_step(limit):
    runs = []
    for own in (True, False):
        bag = Bag([5, 4097])
        runs.append(_step(bag, _optimizer(bag), limit, own)[1])
    assert runs[0] == runs[1]


def test_only_held_gradients_are_written():
    from minitrain_amd.train.update import plan

    bag = Bag([4097, 4097])
    opt = _optimizer(bag)

    def backward():
        sum((p * g).sum() for p, g in zip(bag.p, bag.grads)).backward()

    backward()
    opt.step()
    opt.zero_grad(set_to_none=True)
    backward()
    held = bag.p[0].grad
    update = plan(bag, opt, torch.ones((), device="cuda"), 1.0)
    norm = update.norm(1.0, torch.ones((), device="cuda"))
    update.apply(norm, True)
    torch.testing.assert_close(held, bag.grads[0] * norm[1], rtol=1e-6, atol=0)   # a rounding of the product
    assert torch.equal(bag.p[1].grad, bag.grads[1])
