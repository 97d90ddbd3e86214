"""The decoder's dense operators where something other than a plain first-order pass wants their gradients: function
transforms, forward mode, dispatch modes and gradients of gradients give what the stock operators give (GPU, fp32)."""

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from minitrain_amd.kernels.dense_ops import DenseTorchOps
from minitrain_amd.kernels.hip import HipOpsBackend, dense
from minitrain_amd.model.decoder import layer_means, total_loss
from tests.helpers import hip_backend

pytestmark = pytest.mark.gpu

STOCK = DenseTorchOps()
TOL = dict(rtol=2e-5, atol=2e-5)   # fp32 sums of at most 64 terms of order one, in another order


def _operands(name):
    g = torch.Generator().manual_seed(5)
    r = lambda *shape: torch.randn(*shape, generator=g).cuda()
    if name == "rmsnorm":
        return (r(6, 64), 1 + 0.1 * r(64)), lambda ops, x, w: ops.rmsnorm(x, w, 1e-5)
    if name == "add_rmsnorm":
        def both(ops, x, residual, w):
            if hasattr(ops, "add_rmsnorm"):
                return torch.cat(ops.add_rmsnorm(x, residual, w, 1e-5))
            total = x + residual
            return torch.cat((total, ops.rmsnorm(total, w, 1e-5)))
        return (r(6, 64), r(6, 64), 1 + 0.1 * r(64)), both
    if name == "cross_entropy":
        targets = torch.tensor([1, 0, -100, 6, 3, 3], device="cuda")
        return (r(6, 7),), lambda ops, x: ops.cross_entropy(x, targets)
    if name == "embedding":
        ids = torch.tensor([[1, 0, 4, 1], [2, 1, 4, 4]], device="cuda")

        def lookup(ops, table):
            x = ops.embedding(ids, table, torch.float32) if hasattr(ops, "embedding") else None
            return torch.nn.functional.embedding(ids, table) if x is None else x
        return (r(5, 8),), lookup
    if name == "layer_means":
        return (r(1)[0], r(1)[0], r(1)[0], r(1)[0]), lambda ops, a, b, c, d: torch.stack(layer_means([[a, b], [c, d]], [], ops))
    if name == "total_loss":
        return (r(1)[0], r(1)[0], r(1)[0]), lambda ops, *a: total_loss(*a, 0.25, 0.5, ops)[0]
    angle = r(5, 8)
    cos, sin = angle.cos(), angle.sin()
    if name == "rope":
        return (r(2, 3, 5, 8), r(2, 3, 5, 8)), lambda ops, q, k: torch.stack(ops.rope(q, k, cos, sin))

    def packed(ops, qkv):
        if hasattr(ops, "qkv_rope"):
            turned = ops.qkv_rope(qkv, cos, sin, 3)
            if turned is not None:
                return torch.stack(turned)
        q, k, v = (t.view(2, 5, 3, 8).transpose(1, 2) for t in qkv.chunk(3, dim=-1))
        return torch.stack((*ops.rope(q, k, cos, sin), v))
    return (r(2, 5, 72),), packed


NAMES = ["rmsnorm", "add_rmsnorm", "cross_entropy", "rope", "qkv_rope", "embedding", "layer_means", "total_loss"]


@pytest.mark.parametrize("name", NAMES)
def test_gradients_of_gradients(name):
    print(name, flush=True)
    operands, f = _operands(name)
    results = []
    for ops in (hip_backend(), STOCK):
        leaves = [t.clone().requires_grad_(True) for t in operands]
        out = f(ops, *leaves)
        seed = torch.linspace(-1, 1, out.numel(), device="cuda").reshape(out.shape).requires_grad_(True)
        first = torch.autograd.grad((out.square() * seed).sum(), leaves, create_graph=True)
        second = torch.autograd.grad(sum((t * t).sum() for t in first), [*leaves, seed])
        results.append([*first, *second])
    for got, want in zip(*results):
        torch.testing.assert_close(got, want, rtol=2e-4, atol=2e-4)   # products of up to five factors of order one to ten


@pytest.mark.parametrize("name", NAMES)
def test_function_transforms(name):
    print(name, flush=True)
    operands, f = _operands(name)
    ops = hip_backend()
    tangents = tuple(torch.ones_like(t) for t in operands)
    got, want = (torch.func.jvp(lambda *a: f(o, *a), operands, tangents) for o in (ops, STOCK))
    torch.testing.assert_close(got, want, **TOL)
    got, want = (torch.func.grad(lambda *a: f(o, *a).square().sum())(*operands) for o in (ops, STOCK))
    torch.testing.assert_close(got, want, rtol=1e-4, atol=1e-4)
    stacked = torch.stack([operands[0], 2 * operands[0]])
    got, want = (torch.func.vmap(lambda x: f(o, x, *operands[1:]))(stacked) for o in (ops, STOCK))
    torch.testing.assert_close(got, want, **TOL)


@pytest.mark.parametrize("name", NAMES)
def test_modes_see_the_stock_operators(name):
    print(name, flush=True)
    operands, f = _operands(name)

    class Seen(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    runs = []
    for ops in (hip_backend(), STOCK):
        seen = []
        with Seen():
            f(ops, *operands)
        runs.append(seen)
    assert runs[0] == runs[1]


def test_more_rows_than_one_launch_takes():
    """A launch holds fewer than 2^32 threads; the predicates look at sizes only (tensors of one element, expanded)."""
    one = torch.ones(1, 1, device="cuda")
    w = torch.ones(4, device="cuda")
    assert dense.is_rmsnorm_supported(one.expand(2**26 - 1, 4), w) and not dense.is_rmsnorm_supported(one.expand(2**26, 4), w)
    targets = torch.zeros(1, dtype=torch.long, device="cuda")
    for rows, fits in ((2**23 - 1, True), (2**23, False)):
        assert dense.is_cross_entropy_supported(one.expand(rows, 4), targets.expand(rows)) is fits
    table = torch.ones(2**20, 2, device="cuda")
    for batch, fits in ((2**12 - 1, True), (2**12, False)):
        assert dense.is_qkv_rope_supported(one.view(1, 1, 1).expand(batch, 2**20, 6), table, table, 1) is fits


def test_overridden_operator_is_called():
    class Doubled(HipOpsBackend):
        def rmsnorm(self, x, weight, eps):
            return 2 * super().rmsnorm(x, weight, eps)

        def rope(self, q, k, cos, sin):
            return k, q

    (x, r, w), _ = _operands("add_rmsnorm")
    ops = Doubled()
    torch.testing.assert_close(ops.add_rmsnorm(x, r, w, 1e-5)[1], 2 * STOCK.rmsnorm(x + r, w, 1e-5), **TOL)
    (qkv,), _ = _operands("qkv_rope")
    assert ops.qkv_rope(qkv, torch.ones(5, 8, device="cuda"), torch.ones(5, 8, device="cuda"), 3) is None


def _more_operands(name):
    """The operators that take 16-bit operands only, and the projection of many experts."""
    if name in NAMES:
        return _operands(name)
    g = torch.Generator().manual_seed(6)
    r = lambda *shape: torch.randn(*shape, generator=g).cuda()
    if name == "attention":
        return tuple(r(2, 3, 9, 64).bfloat16() for _ in range(3)), lambda ops, q, k, v: ops.attention(q, k, v, is_causal=True, dropout_p=0.0)
    if name == "qkv_attention":
        angle = r(9, 64)
        cos, sin = angle.cos().bfloat16(), angle.sin().bfloat16()
        return (r(2, 9, 3 * 3 * 64).bfloat16(),), lambda ops, qkv: ops.qkv_attention(qkv, cos, sin, 3, is_causal=True, dropout_p=0.0)
    if name == "linear":
        def project(ops, x, w):
            with torch.autocast("cuda", dtype=torch.bfloat16):
                y = ops.linear(x, w) if hasattr(ops, "linear") else None
                return torch.nn.functional.linear(x, w) if y is None else y
        return (r(2, 520, 64).bfloat16(), r(72, 64) / 8), project
    return (r(37, 64), r(24, 64) / 8), lambda ops, x, w: ops.router_logits(x, w)


# relative to the largest value: fp32 sums of at most 64 terms, or one rounding to bf16 of results whose sums carry others
SCALED_TOL = {torch.float32: 2e-5, torch.bfloat16: 2.0 ** -6}


@pytest.mark.parametrize("name", [*NAMES, "attention", "qkv_attention", "linear", "router_logits"])
@pytest.mark.parametrize("how", ["is_grads_batched", "vmap"])
def test_batched_gradients(name, how):
    """Several gradients of one result in a call, as a vectorised jacobian takes them, against one call for each."""
    print(name, how, flush=True)
    operands, f = _more_operands(name)
    leaves = [t.clone().requires_grad_(True) for t in operands]
    out = f(hip_backend(), *leaves)
    seeds = torch.randn(3, *out.shape, generator=torch.Generator().manual_seed(7)).to(out.dtype).cuda()
    if how == "vmap":
        got = torch.func.vmap(lambda s: torch.autograd.grad(out, leaves, s, retain_graph=True))(seeds)
    else:
        got = torch.autograd.grad(out, leaves, seeds, retain_graph=True, is_grads_batched=True)
    each = [torch.autograd.grad(out, leaves, s, retain_graph=True) for s in seeds]
    for i, (a, leaf) in enumerate(zip(got, leaves)):
        want = torch.stack([e[i] for e in each])
        assert a.dtype == leaf.dtype and a.shape == want.shape
        err, scale = float((a.float() - want.float()).abs().max()), float(want.float().abs().max())
        assert err <= SCALED_TOL[leaf.dtype] * scale, (i, err, scale)


class Through(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def _predicates():
    from minitrain_amd.kernels.hip import is_router_logits_supported
    from minitrain_amd.kernels.hip.moe_layer import moe_layer_violation

    def linear(x, w):
        with torch.autocast("cuda", dtype=torch.bfloat16):
            return dense.is_linear_supported(x, w)

    def layer(w_r, *operands):
        return moe_layer_violation(operands[0], w_r, *operands[1:], 2) is None

    r = lambda *shape: torch.randn(*shape, device="cuda")
    yield "attention", dense.is_attention_supported, [r(2, 3, 9, 64).bfloat16() for _ in range(3)]
    yield "linear", linear, [r(2, 520, 64).bfloat16(), r(72, 64).requires_grad_(True)]
    yield "router_logits", is_router_logits_supported, [r(37, 64), r(24, 64)]
    yield "moe_layer", layer, [r(4, 64), r(37, 64), r(4, 128, 64), r(4, 64, 64)]
    ids = torch.tensor([1, 0, 4], device="cuda")
    yield "embedding", lambda table: dense.is_embedding_supported(ids, table, torch.bfloat16), [r(5, 8).requires_grad_(True)]
    cos, sin = r(9, 64).bfloat16(), r(9, 64).bfloat16()
    yield "qkv_attention", lambda qkv: dense.is_qkv_attention_supported(qkv, cos, sin, 3), [r(2, 9, 3 * 3 * 64).bfloat16()]
    yield "layer_means", lambda a, b, c: dense.is_layer_means_supported([[a, b], [c]], 1), [r(1)[0], r(1)[0], r(1)[0]]
    yield "total_loss", dense.is_total_loss_supported, [r(1)[0], r(1)[0], r(1)[0]]


@pytest.mark.parametrize("which", range(8))
def test_kernels_stay_out_where_somebody_looks(which):
    """The operators that take 16-bit operands only and the layer as one node: not under a transform, a mode or with duals."""
    import torch.autograd.forward_ad as fwd

    name, takes, operands = list(_predicates())[which]
    print(name, flush=True)
    assert takes(*operands)
    answers = []

    def look(first, *others):
        answers.append(takes(first, *others))
        return first.sum()

    first, others = operands[0], operands[1:]
    torch.func.grad(look)(first, *others)
    torch.func.jvp(lambda x: look(x, *others), (first,), (torch.ones_like(first),))
    torch.func.vmap(lambda x: look(x, *others))(torch.stack([first, first]))
    with Through():
        look(*operands)
    with torch.device("cuda"):
        look(*operands)
    with fwd.dual_level():
        look(fwd.make_dual(first, torch.ones_like(first)), *others)
    assert answers == [False] * 6


def test_moe_operators_refuse_transforms():
    """The two MoE operators have no stock form: they raise under a transform and work under a mode."""
    print("MoE operators under transforms", flush=True)
    ops = hip_backend()
    r = lambda *shape: torch.randn(*shape, device="cuda")
    x, w1, w2, logits = r(37, 64), r(4, 128, 64), r(4, 64, 64), r(37, 4)
    route = ops.router_postprocess(logits, 2, normalize=True)
    experts = lambda x: ops.fused_moe(x, w1, w2, route.expert_indices, route.expert_weights)
    weights = lambda l: ops.router_postprocess(l, 2, normalize=True).expert_weights
    for f, operand in ((experts, x), (weights, logits)):
        for transformed in (lambda: torch.func.grad(lambda t: f(t).sum())(operand), lambda: torch.func.vmap(f)(operand.expand(2, *operand.shape)),
                            lambda: torch.func.jvp(f, (operand,), (torch.ones_like(operand),))):
            with pytest.raises(RuntimeError):
                transformed()
        plain = f(operand)
        with Through():
            assert torch.equal(f(operand), plain)
