"""The decoder's dense operators on the GPU against the stock operators of the base backend in fp32.

Tolerances: one rounding of the result to the activation dtype (half an ulp: 2^-9 bf16, 2^-12 fp16 relative to the value),
fp32 sums of at most a few thousand terms elsewhere (1e-5)."""

import pytest
import torch

from minitrain_amd.kernels.dense_ops import DenseTorchOps
from tests.helpers import hip_backend

pytestmark = pytest.mark.gpu

ULP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 1e-5}
STOCK = DenseTorchOps()


def _close(got, want, tol, what, scale=0.0):
    got, want = got.detach().float().cpu(), want.detach().float().cpu()
    scale = max(scale, float(want.abs().max()))
    err = float((got - want).abs().max())
    assert err <= tol * max(scale, 1e-20), (what, err, scale)


@pytest.mark.parametrize("rows,width", [(1, 4), (3, 252), (5, 256), (4099, 768), (130, 1028), (7, 2052), (9, 4096)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("with_residual", [False, True])
def test_rmsnorm(rows, width, dtype, with_residual):
    """One to sixteen groups of four elements per lane, the last one partly empty; more rows than resident waves."""
    print(f"rmsnorm {rows}x{width} {dtype} residual={with_residual}", flush=True)
    ops = hip_backend()
    g = torch.Generator().manual_seed(rows + width)
    x, r, gy, gs = (torch.randn(rows, width, generator=g).to(dtype) for _ in range(4))
    w = 1 + 0.1 * torch.randn(width, generator=g)
    ins = [t.cuda().requires_grad_(True) for t in (x, r, w)]
    ref = [t.double().requires_grad_(True) for t in (x, r, w)]
    if with_residual:
        total, y = ops.add_rmsnorm(ins[0], ins[1], ins[2], 1e-5)
        assert torch.equal(total.cpu(), x + r)
        # the norm is taken of the rounded sum, as it is stored
        want_total = ref[0] + ref[1] + ((x + r).double() - (x.double() + r.double()))
        torch.autograd.backward((total, y), (gs.cuda(), gy.cuda()))
    else:
        y = ops.rmsnorm(ins[0], ins[2], 1e-5)
        want_total = ref[0]
        y.backward(gy.cuda())
    want = want_total * torch.rsqrt(want_total.pow(2).mean(-1, keepdim=True) + 1e-5) * ref[2]
    torch.autograd.backward((want_total, want) if with_residual else (want,), (gs.double(), gy.double()) if with_residual else (gy.double(),))
    assert y.dtype == dtype
    _close(y, want, ULP[dtype], "y")
    _close(ins[0].grad, ref[0].grad, ULP[dtype], "dx")
    if with_residual:
        assert torch.equal(ins[1].grad, ins[0].grad)
    _close(ins[2].grad, ref[2].grad, 1e-5, "dw")   # sums of `rows` fp32 terms


@pytest.mark.parametrize("B,heads,S,D", [(1, 1, 1, 2), (2, 3, 37, 64), (3, 4, 16, 6), (2, 12, 129, 20), (1, 2, 5, 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_rope_and_packed_projection(B, heads, S, D, dtype):
    """Half heads of one, two, four and eight elements per access; separate tensors and the packed projection give what
    the stock operators give, bit for bit in 16-bit types (fp32: products may be contracted), gradients included."""
    print(f"rope B={B} heads={heads} S={S} D={D} {dtype}", flush=True)
    ops = hip_backend()
    g = torch.Generator().manual_seed(S + D)
    qkv, grads = torch.randn(B, S, 3 * heads * D, generator=g).to(dtype), [torch.randn(B, heads, S, D, generator=g).to(dtype).cuda() for _ in range(3)]
    angle = torch.rand(S, D, generator=g) * 6.3
    cos, sin = angle.cos().to(dtype).cuda(), angle.sin().to(dtype).cuda()

    def split(t):
        return (p.view(B, S, heads, D).transpose(1, 2) for p in t.chunk(3, dim=-1))

    def stock(t):
        q, k, v = split(t)
        return (*STOCK.rope(q, k, cos, sin), v)

    def separate(t):
        q, k, v = split(t)
        return (*ops.rope(q, k, cos, sin), v)

    got = {}
    for name, fn in (("stock", stock), ("separate", separate), ("packed", lambda t: ops.qkv_rope(t, cos, sin, heads))):
        leaf = qkv.cuda().requires_grad_(True)
        out = fn(leaf)
        torch.autograd.backward(out, grads)
        got[name] = [*(t.detach() for t in out), leaf.grad]
    for name in ("separate", "packed"):
        for a, b in zip(got[name], got["stock"]):
            if dtype == torch.float32:
                _close(a, b, 1e-6, name)
            else:
                assert torch.equal(a, b), name


@pytest.mark.parametrize("N,V", [(1, 1), (2, 7), (3, 8), (5, 4097), (64, 16385), (33, 50257)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_cross_entropy(N, V, dtype):
    """Rows that start on every alignment, rows shorter than a block, ignored targets; a large maximum and -inf logits."""
    print(f"cross entropy {N}x{V} {dtype}", flush=True)
    ops = hip_backend()
    g = torch.Generator().manual_seed(N + V)
    logits = (4 * torch.randn(N, V, generator=g)).to(dtype)
    targets = torch.randint(0, V, (N,), generator=g)
    if N > 2:
        targets[1] = -100
        logits[0, 0] = 200.0
        logits[2, V // 2] = float("-inf") if targets[2] != V // 2 else 0.0
    leaf = logits.cuda().requires_grad_(True)
    loss = ops.cross_entropy(leaf, targets.cuda())
    (3.0 * loss).backward()
    ref = logits.double().requires_grad_(True)
    want = torch.nn.functional.cross_entropy(ref, targets)
    (3.0 * want).backward()
    assert loss.dtype == torch.float32 and leaf.grad.dtype == dtype
    assert abs(loss.item() - want.item()) <= 1e-5 * max(1.0, abs(want.item()))
    # (a gradient is the difference of a probability and 1: errors are relative to 1 times the factor, also where they cancel)
    _close(leaf.grad, ref.grad, ULP[dtype], "d_logits", scale=3.0 / int((targets != -100).sum()))
    if N > 2:
        assert not leaf.grad[1].any()


def test_cross_entropy_without_valid_targets_and_outside_the_vocabulary():
    ops = hip_backend()
    logits = torch.randn(3, 9, device="cuda")
    assert torch.isnan(ops.cross_entropy(logits, torch.full((3,), -100, device="cuda")))
    assert torch.isnan(ops.cross_entropy(logits, torch.tensor([0, 9, 1], device="cuda")))


@pytest.mark.parametrize("create_graph", [False, True])
def test_gradient_of_targets_outside_the_vocabulary(create_graph):
    """NaN in the rows whose loss is NaN (2^32 + 1 has the low bits of a target inside), what they were in the others."""
    print(f"targets outside the vocabulary, create_graph={create_graph}", flush=True)
    logits = torch.randn(5, 9, device="cuda", requires_grad=True)
    targets = torch.tensor([0, 9, -100, 2 ** 32 + 1, -1], device="cuda")
    d, = torch.autograd.grad(hip_backend().cross_entropy(logits, targets), logits, create_graph=create_graph)
    assert d[[1, 3, 4]].isnan().all() and not d[2].any()
    want = torch.softmax(logits[0].detach(), 0)
    want[0] -= 1
    _close(d[0], want / 4, 1e-5, "row inside", scale=0.25)


def test_results_may_be_changed_in_place():
    """The loss, rotated queries and keys and the attention's result are tensors of their own, as the stock operators' are."""
    print("results changed in place", flush=True)
    g = torch.Generator().manual_seed(2)
    logits, targets = torch.randn(6, 9, generator=g).bfloat16().cuda(), torch.randint(0, 9, (6,), generator=g).cuda()
    q, k, v = (torch.randn(2, 3, 5, 64, generator=g).bfloat16().cuda() for _ in range(3))
    angle = torch.rand(5, 64, generator=g) * 6.3
    cos, sin = angle.cos().bfloat16().cuda(), angle.sin().bfloat16().cuda()
    got = []
    for ops in (hip_backend(), STOCK):
        a, b, c = (t.clone().requires_grad_(True) for t in (logits, q, k))
        loss = ops.cross_entropy(a, targets)
        loss.detach().mul_(3)   # as a logged copy that is reduced over ranks
        loss /= 3
        rotated = ops.rope(b, c, cos, sin)
        for t in rotated:
            t *= 2
        torch.autograd.backward((loss, *rotated), (torch.ones_like(loss), q, k))
        got.append([loss.detach(), *(t.detach() for t in rotated), a.grad, b.grad, c.grad])
    for i, (a, b) in enumerate(zip(*got)):
        _close(a, b, 1e-6 if i == 0 else ULP[torch.bfloat16], i)
    packed = torch.cat([t.transpose(1, 2).reshape(2, 5, -1) for t in (q, k, v)], -1).requires_grad_(True)
    out = hip_backend().attention(*(t.detach().requires_grad_(True) for t in (q, k, v)), is_causal=True, dropout_p=0.0)
    for t in (*hip_backend().qkv_rope(packed, cos, sin, 3)[:2], out):
        t *= 2
