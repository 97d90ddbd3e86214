"""Router projection of more than 16 experts, and the layer node on top of it, at the edges of the tiles."""

import pytest
import torch

from oracle import moe_oracle as O
from tests.helpers import BF16_TOL, assert_close_scaled, hip_backend

pytestmark = pytest.mark.gpu

ULP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 1e-5}


@pytest.mark.parametrize("T,H,E", [(1, 4, 17), (33, 60, 18), (257, 768, 64), (64, 64, 65), (1000, 132, 130), (70, 8192, 24), (4096, 1024, 64)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_wide_projection(T, H, E, dtype):
    """fp32 sums of up to 8192 products of either sign: 1e-5 of the largest value; dx is rounded to the activation dtype."""
    print(f"wide projection T={T} H={H} E={E} {dtype}", flush=True)
    g = torch.Generator().manual_seed(T + E)
    x, w, go = torch.randn(T, H, generator=g).to(dtype), torch.randn(E, H, generator=g) * 0.02, torch.randn(T, E, generator=g)
    a, b = x.cuda().requires_grad_(True), w.cuda().requires_grad_(True)
    y = hip_backend().router_logits(a, b)
    y.backward(go.cuda())
    assert y.dtype == torch.float32 and a.grad.dtype == dtype
    assert_close_scaled(y.detach(), x.double() @ w.double().T, 1e-5, "logits")
    assert_close_scaled(a.grad, go.double() @ w.double(), ULP[dtype], "dx")
    assert_close_scaled(b.grad, go.double().T @ x.double(), 1e-5, "dW")


def _misaligned(t):
    """A dense copy that starts one element behind a 16-byte boundary."""
    return torch.empty(t.numel() + 8, dtype=t.dtype, device="cuda")[1:1 + t.numel()].copy_(t.flatten()).view(t.shape)


def test_operands_that_start_anywhere():
    """The library product that this projection stands in for takes any alignment."""
    print("wide projection, misaligned", flush=True)
    ops = hip_backend()
    x, w_r, w1, w2, g = (t.cuda() for t in O.make_inputs(3, 100, 64, 24, 32))
    results = []
    for place in (lambda t: t.clone(), _misaligned):
        leaves = [place(x).requires_grad_(True), place(w_r).requires_grad_(True), w1.clone().requires_grad_(True), w2.clone().requires_grad_(True)]
        out = ops.moe_layer(*leaves, 4, normalize=True)[0]
        out.backward(g)
        logits = ops.router_logits(leaves[0], leaves[1])
        results.append([out.detach(), logits.detach(), *(t.grad for t in leaves)])
    for a, b in zip(*results):
        assert torch.equal(a, b)


def test_gradient_that_starts_anywhere():
    """Logits of two batches joined: the second part's gradient is a dense slice of the joined one."""
    print("wide projection, misaligned gradient", flush=True)
    ops = hip_backend()
    x, w = torch.randn(5, 64, device="cuda", requires_grad=True), torch.randn(18, 64, device="cuda", requires_grad=True)
    seed = torch.randn(10, 18, device="cuda")
    for rows in (3, 5):   # 54 and 90 elements in front of the slice
        joined = torch.cat((ops.router_logits(x[:rows], w), ops.router_logits(x, w)))
        got = torch.autograd.grad(joined, (x, w), seed[:rows + 5])
        first, second = seed[:rows].double(), seed[rows:rows + 5].double()
        dx = second @ w.double()
        dx[:rows] += first @ w.double()
        assert_close_scaled(got[0], dx, 1e-5, "dx")
        assert_close_scaled(got[1], first.T @ x[:rows].double() + second.T @ x.double(), 1e-5, "dW")


@pytest.mark.parametrize("T,H,E,I,K,capacity", [(500, 128, 24, 64, 2, None), (1000, 256, 64, 128, 4, None), (300, 64, 130, 64, 8, None), (1000, 128, 32, 64, 4, 60)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_layer_node_of_many_experts(T, H, E, I, K, capacity, dtype):
    """One node against the separate operators: the same kernels in the same order up to the sum of the two gradients of x."""
    print(f"layer of many experts T={T} E={E} K={K} capacity={capacity} {dtype}", flush=True)
    ops = hip_backend()
    x, w_r, w1, w2, g = O.make_inputs(T + E, T, H, E, I)
    seeds = (g.to(dtype).cuda(), torch.tensor(0.01, device="cuda"), torch.tensor(0.001, device="cuda"))

    def leaves():
        return [t.cuda().requires_grad_(True) for t in (x.to(dtype), w_r, w1.to(dtype), w2.to(dtype))]

    one, three = leaves(), leaves()
    res = ops.moe_layer(*one, K, normalize=True, **({} if capacity is None else {"capacity": capacity}))
    torch.autograd.backward(res[:3], seeds)
    route = ops.router_postprocess(ops.router_logits(three[0], three[1]), K, normalize=True)
    index, weights = route.expert_indices, route.expert_weights
    if capacity is not None:
        keep, index, _ = ops.capacity_mask(index, weights, E, capacity)
        weights = weights * keep
        total = weights.sum(-1, keepdim=True)
        weights = torch.where(total > 0, weights / total.clamp_min(torch.finfo(torch.float32).eps), weights)
    out = ops.fused_moe(three[0], three[2], three[3], index, weights.to(dtype))
    torch.autograd.backward((out, route.load_balance_loss, route.z_loss), seeds)
    tol = 1e-5 if dtype == torch.float32 else BF16_TOL
    assert_close_scaled(res[0].detach(), out.detach(), tol, "out")
    torch.testing.assert_close(res[1], route.load_balance_loss, rtol=2e-5, atol=1e-7)
    for name, a, b in zip(("dx", "dW_r", "dW1", "dW2"), one, three):
        assert_close_scaled(a.grad, b.grad, tol, name)
