"""Rotary encoding and attention of a packed projection as one node: what the separate operators give, and fp64.

The result is theirs bit for bit.  The gradients of queries and keys are rounded once where the separate operators round them, then the products of the
turn back and then their sum: 2 * 2^-7 (2^-10) of the largest value as in the attention's own tests, and within that against fp64."""

import pytest
import torch

from minitrain_amd.kernels.hip import HipOpsBackend
from tests.helpers import hip_backend
from tests.test_gpu_attention import TOL, _close, _written_out

pytestmark = pytest.mark.gpu


def _operands(B, heads, S, dtype, seed=0):
    g = torch.Generator().manual_seed(S + heads + seed)
    qkv, grad = torch.randn(B, S, 3 * heads * 64, generator=g).to(dtype).cuda(), torch.randn(B, S, heads * 64, generator=g).to(dtype).cuda()
    angle = torch.rand(S, 64, generator=g) * 6.3   # halves of their own
    return qkv, angle.cos().to(dtype).cuda(), angle.sin().to(dtype).cuda(), grad


def _separate(ops, qkv, cos, sin, heads, causal):
    q, k, v = ops.qkv_rope(qkv, cos, sin, heads)
    out = ops.attention(q, k, v, is_causal=causal, dropout_p=0.0)
    return out.transpose(1, 2).reshape(qkv.shape[0], qkv.shape[1], -1)


def _wide(qkv, cos, sin, heads, causal):
    q, k, v = (t.view(*t.shape[:2], heads, 64).transpose(1, 2) for t in qkv.chunk(3, -1))
    turn = lambda t: t * cos + torch.cat((-t[..., 32:], t[..., :32]), -1) * sin
    return _written_out(turn(q), turn(k), v, causal).transpose(1, 2).reshape(qkv.shape[0], qkv.shape[1], -1)


@pytest.mark.parametrize("B,heads,S", [(1, 1, 1), (2, 3, 31), (1, 9, 65), (2, 12, 128), (1, 5, 129), (1, 2, 777), (1, 3, 1024)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("causal", [True, False])
def test_one_node(B, heads, S, dtype, causal):
    print(f"qkv attention B={B} heads={heads} S={S} {dtype} causal={causal}", flush=True)
    ops = hip_backend()
    qkv, cos, sin, grad = _operands(B, heads, S, dtype)
    leaf, other, ref = (qkv.clone().requires_grad_(True), qkv.clone().requires_grad_(True), qkv.double().requires_grad_(True))
    out = ops.qkv_attention(leaf, cos, sin, heads, is_causal=causal, dropout_p=0.0)
    want = _separate(ops, other, cos, sin, heads, causal)
    assert torch.equal(out, want) and out.is_contiguous()
    with torch.no_grad():
        assert torch.equal(ops.qkv_attention(leaf, cos, sin, heads, is_causal=causal, dropout_p=0.0), want)
    out.backward(grad)
    want.backward(grad)
    exact = _wide(ref, cos.double(), sin.double(), heads, causal)
    exact.backward(grad.double())
    # scores of turned and rounded queries and keys: half an ulp of each on 64 products, 2^-9 * sqrt(2 / 64) * |q| |k| / 8 < 2^-7 of a probability
    for part in range(3):
        pick = slice(part * heads * 64, (part + 1) * heads * 64)
        _close(leaf.grad[..., pick], other.grad[..., pick].double(), 2 * TOL[dtype], f"gradient {part}")
        mine, theirs = (float((t.grad[..., pick].double() - ref.grad[..., pick]).norm()) for t in (leaf, other))
        assert mine <= 1.02 * theirs + 64 * 2.0 ** -24, (part, mine, theirs)   # one rounding in the place of three


@pytest.mark.parametrize("layout", ["misaligned", "one value", "rows apart"])
def test_layouts(layout):
    ops = hip_backend()
    qkv, cos, sin, grad = _operands(2, 3, 70, torch.bfloat16)
    if layout == "misaligned":
        qkv = torch.cat((qkv[..., :1], qkv), -1)[..., 1:]
    grad = torch.ones((), device="cuda", dtype=torch.bfloat16).expand(grad.shape) if layout == "one value" else torch.cat((grad, grad), -1)[..., :192]
    results = []
    for f in (lambda t: ops.qkv_attention(t, cos, sin, 3, is_causal=True, dropout_p=0.0), lambda t: _separate(ops, t, cos, sin, 3, True)):
        leaf = qkv.detach().requires_grad_(True)
        out = f(leaf)
        out.backward(grad)
        results.append((out.detach(), leaf.grad))
    assert torch.equal(results[0][0], results[1][0])
    _close(results[0][1], results[1][1].double(), 2 * TOL[torch.bfloat16], "gradient")


def test_other_calls_stay_with_the_separate_operators():
    ops = hip_backend()
    qkv, cos, sin, _ = _operands(1, 2, 40, torch.bfloat16)
    call = lambda backend, t=qkv, c=cos, heads=2, p=0.0: backend.qkv_attention(t, c, sin, heads, is_causal=True, dropout_p=p)
    assert call(ops) is not None
    assert call(ops, p=0.1) is None and call(ops, heads=4) is None and call(ops, c=cos[:20]) is None and call(ops, t=qkv.float()) is None
    with torch.nn.attention.sdpa_kernel(torch.nn.attention.SDPBackend.MATH):
        assert call(ops) is None
    with torch.autocast("cuda", dtype=torch.float16):
        assert call(ops) is None

    class Own(HipOpsBackend):
        def attention(self, q, k, v, *, is_causal, dropout_p):
            return super().attention(q, k, v, is_causal=is_causal, dropout_p=dropout_p)

    assert call(Own()) is None


def test_gradient_of_a_gradient():
    ops = hip_backend()
    qkv, cos, sin, _ = _operands(1, 2, 9, torch.bfloat16)
    results = []
    for f, leaf in ((lambda t: ops.qkv_attention(t, cos, sin, 2, is_causal=True, dropout_p=0.0), qkv.requires_grad_(True)),
                    (lambda t: _wide(t, cos.double(), sin.double(), 2, True), qkv.detach().double().requires_grad_(True))):
        first, = torch.autograd.grad(f(leaf).square().sum(), leaf, create_graph=True)
        results.append(torch.autograd.grad(first.square().sum(), leaf)[0])
    _close(results[0], results[1], 2.0 ** -4, "second derivative")   # a chain of six bf16 roundings, each amplified by a factor of up to two
