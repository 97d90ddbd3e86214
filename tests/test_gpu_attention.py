"""Attention of heads of 64 elements on the GPU against the same products written out in fp64.

Tolerances, relative to the largest value of a result: one rounding of it to the 16-bit type (half an ulp, 2^-9 or 2^-12)
and one of each probability or score gradient that enters its sum (independent, so well under a further ulp): 2^-7 and 2^-10.
The gradients carry the rounding of the output through delta as well: twice that.  With a single key dP and delta cancel to
the rounding of two fp32 sums of 64 products of order one: 64 * 2^-24 on top."""

import pytest
import torch

from minitrain_amd.kernels.dense_ops import DenseTorchOps
from minitrain_amd.kernels.hip import dense
from tests.helpers import hip_backend

pytestmark = pytest.mark.gpu

TOL = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}


def _written_out(q, k, v, causal):
    score = q @ k.transpose(-1, -2).contiguous() * 0.125
    if causal:
        score = score.masked_fill(torch.ones(q.shape[2], q.shape[2], dtype=torch.bool, device=q.device).triu(1), float("-inf"))
    return torch.softmax(score, -1) @ v


def _close(got, want, tol, what):
    err, scale = float((got.double().cpu() - want.cpu()).abs().max()), float(want.abs().max())
    assert err <= tol * scale + 64 * 2.0 ** -24, (what, err, scale)


@pytest.mark.parametrize("B,heads,S", [(1, 1, 1), (2, 3, 31), (1, 9, 64), (3, 4, 65), (2, 12, 128), (1, 5, 129), (2, 12, 200), (1, 2, 777), (1, 3, 1024)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("causal", [True, False])
def test_attention(B, heads, S, dtype, causal):
    """Partly filled tiles of queries and keys, one block and several, head counts that do not fill the XCDs evenly; queries,
    keys and values as views of one projection, the gradient in the layout that the output projection leaves."""
    print(f"attention B={B} heads={heads} S={S} {dtype} causal={causal}", flush=True)
    g = torch.Generator().manual_seed(S + heads)
    packed = torch.randn(B, S, 3, heads, 64, generator=g).to(dtype).cuda()
    q, k, v = (packed[:, :, i].transpose(1, 2).detach().requires_grad_(True) for i in range(3))
    grad = torch.randn(B, S, heads, 64, generator=g).to(dtype).cuda().transpose(1, 2)
    ref = [t.detach().double().requires_grad_(True) for t in (q, k, v)]
    assert dense.is_attention_supported(q, k, v)
    out = hip_backend().attention(q, k, v, is_causal=causal, dropout_p=0.0)
    assert out.dtype == dtype and out.shape == q.shape
    out.backward(grad)
    want = _written_out(*ref, causal)
    want.backward(grad.double())
    _close(out.detach(), want.detach(), TOL[dtype], "out")
    for got, w, what in zip((q, k, v), ref, ("dq", "dk", "dv")):
        _close(got.grad, w.grad, 2 * TOL[dtype], what)


def test_large_scores_and_rows_without_a_finite_score():
    """Scores far apart (a probability of one), a row that sees only -inf (not a number, as in the stock operator)."""
    print("attention, large scores", flush=True)
    g = torch.Generator().manual_seed(1)
    q, k, v = (torch.randn(1, 2, 150, 64, generator=g).bfloat16().cuda() for _ in range(3))
    q, k = 40 * q, 40 * k   # scores of some thousands, whose fp32 sums are good to about 2^-24 * 64 * 1600 / 8 < 2^-10
    out = hip_backend().attention(q, k, v, is_causal=True, dropout_p=0.0)
    _close(out, _written_out(q.double(), k.double(), v.double(), True), TOL[torch.bfloat16], "out")
    q[0, 0, 3], k[0, 0, :4] = 1.0, float("-inf")
    out = hip_backend().attention(q.abs(), k, v, is_causal=True, dropout_p=0.0)
    assert out[0, 0, :4].isnan().all() and out[0, 0, 4:].isfinite().all() and out[0, 1].isfinite().all()


def _layouts():
    g = torch.Generator().manual_seed(9)
    r = lambda *shape: torch.randn(*shape, generator=g).bfloat16().cuda()
    yield "heads in front", [r(3, 2, 70, 64).transpose(0, 1) for _ in range(3)]
    yield "rows in front", [r(70, 2, 3, 64).permute(1, 2, 0, 3) for _ in range(3)]
    yield "one batch for all", [r(1, 3, 70, 64).expand(2, 3, 70, 64) for _ in range(3)]
    yield "one head for all keys and values", [r(2, 3, 70, 64), r(2, 1, 70, 64).expand(2, 3, 70, 64), r(2, 1, 70, 64).expand(2, 3, 70, 64)]
    yield "every other row", [r(2, 3, 140, 64)[:, :, ::2] for _ in range(3)]
    yield "part of a wider row", [r(2, 3, 70, 136)[..., 8:72] for _ in range(3)]


@pytest.mark.parametrize("which", range(6))
@pytest.mark.parametrize("grad_layout", ["dense", "one value", "rows in front", "misaligned"])
def test_layouts(which, grad_layout):
    """Every order of the outer dimensions, strides of zero, rows apart; gradients as reductions and slices leave them."""
    name, (q, k, v) = list(_layouts())[which]
    print(f"attention, {name}, gradient {grad_layout}", flush=True)
    assert dense.is_attention_supported(q, k, v)
    leaves = [t.detach().requires_grad_(True) for t in (q, k, v)]
    ref = [t.detach().double().requires_grad_(True) for t in (q, k, v)]
    g = torch.Generator().manual_seed(10)
    grad = {"dense": lambda: torch.randn(2, 3, 70, 64, generator=g), "one value": lambda: torch.ones(()).expand(2, 3, 70, 64),
            "rows in front": lambda: torch.randn(70, 3, 2, 64, generator=g).permute(2, 1, 0, 3),
            "misaligned": lambda: torch.randn(2, 3, 70, 65, generator=g)}[grad_layout]().bfloat16().cuda()
    grad = grad[..., 1:] if grad_layout == "misaligned" else grad
    out = hip_backend().attention(*leaves, is_causal=True, dropout_p=0.0)
    out.backward(grad)
    want = _written_out(*ref, True)
    want.backward(grad.double())
    _close(out.detach(), want.detach(), TOL[torch.bfloat16], "out")
    for got, w, what in zip(leaves, ref, ("dq", "dk", "dv")):
        _close(got.grad, w.grad, 2 * TOL[torch.bfloat16], what)


def test_other_layouts_types_and_choices_stay_stock():
    ops, stock = hip_backend(), DenseTorchOps()
    q = torch.randn(1, 2, 40, 64, device="cuda", dtype=torch.bfloat16)
    assert dense.is_attention_supported(q, q, q)
    odd = torch.randn(1, 2, 40, 65, device="cuda", dtype=torch.bfloat16)[..., 1:]
    for t in (q.float(), q[..., :32], odd, q.transpose(2, 3)):
        assert not dense.is_attention_supported(t, t, t)
    assert not dense.is_attention_supported(q, q[:, :, :7], q[:, :, :7])
    with torch.nn.attention.sdpa_kernel(torch.nn.attention.SDPBackend.MATH):
        assert not dense.is_attention_supported(q, q, q)
    with torch.autocast("cuda", dtype=torch.float16):
        assert not dense.is_attention_supported(q, q, q)
    assert torch.equal(ops.attention(odd, odd, odd, is_causal=True, dropout_p=0.0), stock.attention(odd, odd, odd, is_causal=True, dropout_p=0.0))


def test_gradient_of_a_gradient():
    leaves = [torch.randn(1, 2, 9, 64, device="cuda").bfloat16().requires_grad_(True) for _ in range(3)]
    wide = [t.detach().double().requires_grad_(True) for t in leaves]
    results = []
    for f, ts in ((lambda *a: hip_backend().attention(*a, is_causal=True, dropout_p=0.0), leaves), (lambda *a: _written_out(*a, True), wide)):
        first = torch.autograd.grad(f(*ts).square().sum(), ts, create_graph=True)
        results.append(torch.autograd.grad(sum(t.square().sum() for t in first), ts))
    for got, want in zip(*results):
        _close(got, want, 2.0 ** -5, "second derivative")   # a chain of four bf16 roundings, each amplified by a factor of up to two
