"""Grouped GEMMs with few rows per expert on 128 x 128 tiles: the operator's results and gradients against fp64 (GPU).

Tolerance, relative to the largest value: 2^-7 (bf16) and 2^-10 (fp16), two half-ulp roundings of the intermediates that enter
the last product and one of its result."""

import pytest
import torch

from minitrain_amd.kernels.hip.fused_moe import fused_moe
from tests.helpers import BF16_TOL, assert_close_scaled, hip_moe_grads, oracle_moe_grads, routed_case

pytestmark = pytest.mark.gpu

TOL = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}


@pytest.mark.parametrize("rows,E,H,I", [
    ((127, 128, 129), 3, 256, 256), ((256, 0, 1), 3, 128, 192), ((300, 50), 2, 712, 328), ((95, 400, 96, 33, 0, 64), 6, 768, 512), ((1,), 1, 320, 1368)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("params", ["same", "fp32"])
def test_small_tiles(rows, E, H, I, dtype, params):
    """One row to three tiles of an expert and one more or less, experts without rows, widths that are not whole tiles."""
    print(f"small tiles rows={rows} H={H} I={I} {dtype} {params}", flush=True)
    g = torch.Generator().manual_seed(sum(rows) + H)
    T = sum(rows)
    pt = torch.float32 if params == "fp32" else dtype
    idx = torch.repeat_interleave(torch.arange(E), torch.tensor(rows))[torch.randperm(T, generator=g)].int()[:, None].cuda()
    x, grad = (torch.randn(T, H, generator=g).to(dtype).cuda() for _ in range(2))
    w1, w2 = (torch.randn(E, 2 * I, H, generator=g) * H ** -0.5).to(pt).cuda(), (torch.randn(E, H, I, generator=g) * I ** -0.5).to(pt).cuda()
    s = (0.5 + torch.rand(T, 1, generator=g)).to(dtype).cuda()
    leaves = [t.requires_grad_(True) for t in (x, w1, w2, s)]
    out = fused_moe(x, w1, w2, idx, s)
    out.backward(grad)
    # the weights enter the products in the activation dtype
    wide = [x.detach().double(), w1.detach().to(dtype).double(), w2.detach().to(dtype).double(), s.detach().double()]
    wide = [t.requires_grad_(True) for t in wide]
    parts = []
    for e in range(E):
        at = (idx[:, 0] == e).nonzero()[:, 0]
        gate, up = (wide[0][at] @ wide[1][e].T).chunk(2, dim=1)
        parts.append((at, ((torch.nn.functional.silu(gate) * up) @ wide[2][e].T) * wide[3][at]))
    want = torch.zeros(T, H, dtype=torch.float64, device="cuda").index_copy(0, torch.cat([p[0] for p in parts]), torch.cat([p[1] for p in parts]))
    want.backward(grad.double())
    for what, got, ref in [("out", out.detach(), want.detach())] + [(n, a.grad, b.grad) for n, a, b in zip(("dx", "dw1", "dw2", "ds"), leaves, wide)]:
        err, scale = float((got.double() - ref).abs().max()), float(ref.abs().max())
        assert err <= TOL[dtype] * scale, (what, err, scale)


@pytest.mark.parametrize("T,H,E,I,K", [(2946, 128, 8, 1024, 2), (3400, 72, 16, 1000, 1), (6544, 128, 8, 768, 2), (5122, 64, 16, 680, 3), (5200, 64, 8, 1024, 2)])
def test_gradient_on_large_tiles_within_the_round_of_narrow_ones(T, H, E, I, K):
    """dO*W2 where a CU would hold two or three narrow blocks and the large tiles are half a round, cut in two, or a whole one; and one call that
    stays: the gradients that pass through it."""
    print(f"dO*W2 on large tiles T={T} H={H} E={E} I={I} K={K}", flush=True)
    case = routed_case(31 + T, T, H, E, I, K, bias=torch.linspace(-0.5, 0.5, E))
    _, grads = hip_moe_grads(case["x"], case["w1"], case["w2"], case["idx"], case["w"], case["g"])
    _, ref = oracle_moe_grads(case["x"], case["w1"], case["w2"], case["idx"], case["w"], case["g"], device="cuda")
    for name, a, b in zip(("dx", "dW1", "dW2", "dS"), grads, ref):
        assert_close_scaled(a, b, BF16_TOL, name)


@pytest.mark.parametrize("T,H,E,I,K", [(1600, 768, 8, 1024, 2), (1810, 776, 8, 1024, 2), (5400, 256, 8, 1400, 2), (5700, 256, 8, 1400, 2), (700, 512, 24, 520, 3)])
@pytest.mark.parametrize("fp32_weights", [False, True])
def test_dx_in_front_of_the_weight_gradients(T, H, E, I, K, fp32_weights):
    """The joint backward launch with its dX tiles in front: on both sides of the line to small tiles behind, on both sides of I rows an expert, and
    with ragged widths; an expert without routes, popular ones."""
    print(f"dX in front T={T} H={H} E={E} I={I} K={K} fp32_weights={fp32_weights}", flush=True)
    bias = torch.linspace(-1.0, 1.0, E)
    bias[1] = -100.0
    case = routed_case(37 + T, T, H, E, I, K, bias=bias)
    w1, w2 = ((case[n].float() if fp32_weights else case[n]) for n in ("w1", "w2"))
    _, grads = hip_moe_grads(case["x"], w1, w2, case["idx"], case["w"], case["g"])
    _, ref = oracle_moe_grads(case["x"], case["w1"], case["w2"], case["idx"], case["w"], case["g"], device="cuda")
    for name, a, b in zip(("dx", "dW1", "dW2", "dS"), grads, ref):
        assert_close_scaled(a, b, BF16_TOL, name)
