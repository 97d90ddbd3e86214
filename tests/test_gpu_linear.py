"""Projection under autocast with the weight gradient summed in fp32, against fp64 products of the rounded operands (GPU).

The sum of T products of order one in fp32, in segments: an error of at most sqrt(T) * 2^-24 of its own size with margin, 1e-5
of the largest value for the lengths here.  The other results carry one 16-bit rounding (2^-8, 2^-11)."""

import pytest
import torch

from minitrain_amd import _lib
from minitrain_amd.kernels.hip import dense
from tests.helpers import hip_backend

pytestmark = pytest.mark.gpu

ULP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


@pytest.mark.parametrize("T,N,K", [(1024, 8, 8), (1025, 256, 256), (1600, 264, 248), (4099, 768, 768), (2000, 2304, 768), (9000, 1032, 40), (1500, 1000, 2048)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_linear(T, N, K, dtype):
    """Segments of one k-tile and of several, the last one partly filled, widths that are not whole tiles, one tile and 32."""
    print(f"linear T={T} N={N} K={K} {dtype}", flush=True)
    g = torch.Generator().manual_seed(T)
    x = torch.randn(T, K, generator=g).to(dtype).cuda().requires_grad_(True)
    w = (torch.randn(N, K, generator=g) * K ** -0.5).cuda().requires_grad_(True)
    grad = torch.randn(T, N, generator=g).to(dtype).cuda()
    with torch.autocast("cuda", dtype=dtype):
        y = hip_backend().linear(x, w)
    assert y is not None and y.dtype == dtype
    y.backward(grad)
    wide = w.detach().to(dtype).double()
    for got, want, tol, what in ((y.detach(), x.detach().double() @ wide.T, ULP[dtype], "y"), (x.grad, grad.double() @ wide, ULP[dtype], "dx"),
                                 (w.grad, grad.double().T @ x.detach().double(), 1e-5, "dw")):
        err, scale = float((got.double() - want).abs().max()), float(want.abs().max())
        assert err <= tol * scale, (what, err, scale)
    assert w.grad.dtype == torch.float32


@pytest.mark.parametrize("T", [128, 129, 255, 256, 257, 511, 513, 1023])
@pytest.mark.parametrize("N,K", [(264, 248), (768, 768), (2304, 768)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_linear_of_few_rows(T, N, K, dtype):
    """One segment, whose tiles are the result, and two; products of either kind beside it."""
    test_linear(T, N, K, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_linear_of_fewer_rows_is_the_callers(dtype):
    x, w = torch.randn(127, 768, device="cuda", dtype=dtype, requires_grad=True), torch.randn(768, 768, device="cuda", requires_grad=True)
    assert not _lib.load().mts_linear_dw_supported(_lib.dtype_code(dtype), 127, 768, 768)
    with torch.autocast("cuda", dtype=dtype):
        assert hip_backend().linear(x, w) is None


@pytest.mark.parametrize("T,N,K,pad", [(128, 64, 8, 0), (131, 67, 8, 5), (300, 1003, 120, 21), (1025, 2112, 264, 0), (520, 9001, 1000, 7), (66000, 67, 8, 61), (66000, 64, 8, 8),
                                       (130, 66001, 8, 7)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_linear_in_rounds(T, N, K, pad, dtype):
    """Outputs of at least eight times the input's width: reductions of one k-tile and of many, cut and whole, with every remainder of the
    16-byte chunks; more tiles than the chip has CUs; rows of the gradient that are further apart, with NaN between them."""
    print(f"linear in rounds T={T} N={N} K={K} pad={pad} {dtype}", flush=True)
    g = torch.Generator().manual_seed(T)
    x = torch.randn(T, K, generator=g).to(dtype).cuda().requires_grad_(True)
    w = (torch.randn(N, K, generator=g) * K ** -0.5).cuda().requires_grad_(True)
    rows = torch.full((T, N + pad), float("nan"), dtype=dtype, device="cuda")
    grad = rows[:, :N]
    grad.copy_(torch.randn(T, N, generator=g))
    with torch.autocast("cuda", dtype=dtype):
        y = hip_backend().linear(x, w)
    y.backward(grad)
    wide = w.detach().to(dtype).double()
    for got, want, tol, what in ((x.grad, grad.double() @ wide, ULP[dtype], "dx"), (w.grad, grad.double().T @ x.detach().double(), 1e-5, "dw")):
        err, scale = float((got.double() - want).abs().max()), float(want.abs().max())
        assert err <= tol * scale, (what, err, scale)
    assert w.grad.dtype == torch.float32


@pytest.mark.parametrize("N", [64, 67])
@pytest.mark.parametrize("layout", ["dense", "every other column", "misaligned", "gradient of one value", "nothing behind the last row"])
def test_gradients_in_other_layouts_in_rounds(layout, N):
    """What the kernels read in place and what is copied for them: the same products."""
    print(f"linear in rounds, {layout}, {N} columns", flush=True)
    g = torch.Generator().manual_seed(6)
    r = lambda *shape: torch.randn(*shape, generator=g).bfloat16().cuda()
    grad = {"dense": lambda: r(200, N), "every other column": lambda: r(200, 2 * N)[:, ::2], "misaligned": lambda: r(200, 80)[:, 1:N + 1],
            "gradient of one value": lambda: torch.ones((), device="cuda", dtype=torch.bfloat16).expand(200, N),
            "nothing behind the last row": lambda: r(199 * 72 + N).as_strided((200, N), (72, 1))}[layout]()
    x, w = r(200, 8).requires_grad_(True), torch.randn(N, 8, generator=g).cuda().requires_grad_(True)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = hip_backend().linear(x, w)
    y.backward(grad)
    for got, want in ((x.grad, grad.double() @ w.detach().bfloat16().double()), (w.grad, grad.double().T @ x.detach().double())):
        assert float((got.double() - want).abs().max()) <= ULP[torch.bfloat16] * float(want.abs().max())


@pytest.mark.parametrize("layout", ["sequence first", "part of a wider row", "misaligned", "weight by columns"])
def test_operands_in_other_layouts_in_rounds(layout):
    """Inputs that are not dense or not aligned and a weight that is not: the same gradients."""
    print(f"linear in rounds, {layout}", flush=True)
    g = torch.Generator().manual_seed(7)
    r = lambda *shape: torch.randn(*shape, generator=g).bfloat16().cuda()
    x = {"sequence first": lambda: r(100, 2, 16).transpose(0, 1), "part of a wider row": lambda: r(2, 100, 48)[..., 16:32], "misaligned": lambda: r(2, 100, 17)[..., 1:],
         "weight by columns": lambda: r(2, 100, 16)}[layout]().detach().requires_grad_(True)
    w = torch.randn(16, 136, generator=g).cuda().t() if layout == "weight by columns" else torch.randn(136, 16, generator=g).cuda()
    w = w.detach().requires_grad_(True)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = hip_backend().linear(x, w)
    grad = r(2, 100, 136)
    y.backward(grad)
    wide, rows = w.detach().bfloat16().double(), grad.double().reshape(-1, 136)
    for got, want, tol in ((y.detach(), x.detach().double() @ wide.T, ULP[torch.bfloat16]), (x.grad, grad.double() @ wide, ULP[torch.bfloat16]),
                           (w.grad, rows.T @ x.detach().double().reshape(-1, 16), 1e-5)):
        assert got.shape == want.shape and float((got.double() - want).abs().max()) <= tol * float(want.abs().max())


@pytest.mark.parametrize("create_graph", [False, True])
def test_vocabulary_weight_changed_before_the_backward_pass(create_graph):
    """The gradients are those of the weight of the forward pass, and can be differentiated again."""
    print(f"linear in rounds, weight changed in place, create_graph={create_graph}", flush=True)
    g = torch.Generator().manual_seed(8)
    x, w = torch.randn(2, 100, 16, generator=g).bfloat16().cuda().requires_grad_(True), torch.randn(136, 16, generator=g).cuda().requires_grad_(True)
    grad = torch.randn(2, 100, 136, generator=g).bfloat16().cuda()
    got = []
    for f in (lambda: hip_backend().linear(x, w), lambda: torch.nn.functional.linear(x, w)):
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = f()
        with torch.no_grad():
            w.mul_(2)
        got.append(torch.autograd.grad(y, (x, w), grad, create_graph=create_graph))
        with torch.no_grad():
            w.div_(2)
    for a, b in zip(*got):
        assert a.dtype == b.dtype and a.requires_grad == create_graph and float((a.detach().float() - b.detach().float()).abs().max()) <= ULP[torch.bfloat16] * float(b.detach().abs().max())


@pytest.mark.parametrize("rows,V", [(130, 64), (200, 1003), (129, 50257)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_loss_on_a_projection(rows, V, dtype):
    """The gradient of the logits of a projection has the values that a leaf's has, and is dense where somebody sees it."""
    print(f"loss on a projection {rows}x{V} {dtype}", flush=True)
    g = torch.Generator().manual_seed(V)
    x, w = torch.randn(1, rows, 8, generator=g).to(dtype).cuda().requires_grad_(True), torch.randn(V, 8, generator=g).cuda().requires_grad_(True)
    targets = torch.randint(0, V, (rows,), generator=g).cuda()
    targets[1] = -100
    ops = hip_backend()
    with torch.autocast("cuda", dtype=dtype):
        logits = ops.linear(x, w)
        seen = []
        logits.register_hook(seen.append)
        ops.cross_entropy(logits.reshape(-1, V), targets).backward()
    leaf = logits.detach().view(-1, V).requires_grad_(True)
    ops.cross_entropy(leaf, targets).backward()
    assert torch.equal(seen[0].view(-1, V), leaf.grad) and leaf.grad.is_contiguous()
    assert seen[0].is_contiguous() and logits.is_contiguous()
    for got, want, tol in ((x.grad[0], leaf.grad.double() @ w.detach().to(dtype).double(), ULP[dtype]), (w.grad, leaf.grad.double().T @ x.detach()[0].double(), 1e-5)):
        assert float((got.double() - want).abs().max()) <= tol * float(want.abs().max())


@pytest.mark.parametrize("who", ["hook of the logits", "hook of their view", "retain_grad", "autograd.grad", "hook before the node", "hook behind the node",
                                 "hook behind the loss", "module hook", "nobody"])
def test_who_sees_the_gradient_of_the_logits_sees_it_dense(who):
    """Rows of an odd vocabulary are pitched on their way from the loss to the projection only where nobody can see them; the gradients of
    the projection are the same."""
    print(f"gradient of the logits seen by {who}", flush=True)
    rows, V = 256, 8193
    g = torch.Generator().manual_seed(9)
    x, w = torch.randn(2, rows // 2, 8, generator=g).bfloat16().cuda().requires_grad_(True), torch.randn(V, 8, generator=g).cuda().requires_grad_(True)
    targets = torch.randint(0, V, (rows,), generator=g).cuda()
    ops, seen = hip_backend(), []

    class Head(torch.nn.Module):
        def forward(self, x):
            return ops.linear(x, w)

    head = Head()
    if who == "module hook":
        head.register_full_backward_hook(lambda module, into, out: seen.append(out[0]))
    with torch.autocast("cuda", dtype=torch.bfloat16):
        logits = head(x)
        flat = logits.view(-1, V)
        loss = ops.cross_entropy(flat, targets)
    node = logits.grad_fn
    {"hook of the logits": lambda: logits.register_hook(seen.append), "hook of their view": lambda: flat.register_hook(seen.append), "retain_grad": logits.retain_grad,
     "hook before the node": lambda: node.register_prehook(lambda out: seen.append(out[0])),
     "hook behind the node": lambda: node.register_hook(lambda into, out: seen.append(out[0])),
     "hook behind the loss": lambda: loss.grad_fn.register_hook(lambda into, out: seen.append(into[0]))}.get(who, lambda: None)()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    if who == "autograd.grad":
        *grads, d = torch.autograd.grad(loss, (x, w, logits))
        seen.append(d)
    else:
        loss.backward()
        grads = [x.grad, w.grad]
    if who == "retain_grad":
        seen.append(logits.grad)
    leaf = flat.detach().requires_grad_(True)
    peak = torch.cuda.max_memory_allocated() - before
    ops.cross_entropy(leaf, targets).backward()
    assert len(seen) == (who != "nobody")
    for d in seen:
        assert d.is_contiguous() and torch.equal(d.view(-1), leaf.grad.view(-1))
    # a dense gradient is copied on its way
    assert (peak < 2 * leaf.numel() * 2) == (who == "nobody"), peak
    for got, want, tol in ((grads[0].view(-1, 8), leaf.grad.double() @ w.detach().bfloat16().double(), ULP[torch.bfloat16]),
                           (grads[1], leaf.grad.double().T @ x.detach().double().view(-1, 8), 1e-5)):
        assert float((got.double() - want).abs().max()) <= tol * float(want.abs().max())


@pytest.mark.parametrize("layout", ["sequence first", "every other row", "part of a wider row", "misaligned", "gradient of one value"])
def test_layouts(layout):
    """Operands and gradients that are not dense or not aligned go through a copy: the same sums."""
    print(f"linear, {layout}", flush=True)
    g = torch.Generator().manual_seed(3)
    r = lambda *shape: torch.randn(*shape, generator=g).bfloat16().cuda()
    x = {"sequence first": lambda: r(600, 2, 64).transpose(0, 1), "every other row": lambda: r(2, 1200, 64)[:, ::2], "misaligned": lambda: r(2, 600, 65)[..., 1:],
         "part of a wider row": lambda: r(2, 600, 128)[..., 32:96], "gradient of one value": lambda: r(2, 600, 64)}[layout]()
    w = torch.randn(72, 64, generator=g).cuda().requires_grad_(True)
    x = x.detach().requires_grad_(True)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = hip_backend().linear(x, w)
    grad = torch.ones((), device="cuda", dtype=torch.bfloat16).expand(2, 600, 72) if layout == "gradient of one value" else r(2, 72, 600).transpose(1, 2)
    y.backward(grad)
    wide = w.detach().bfloat16().double()
    for got, want, tol, what in ((y.detach(), x.detach().double() @ wide.T, ULP[torch.bfloat16], "y"), (x.grad, grad.double() @ wide, ULP[torch.bfloat16], "dx"),
                                 (w.grad, grad.double().reshape(-1, 72).T @ x.detach().double().reshape(-1, 64), 1e-5, "dw")):
        err, scale = float((got.double() - want).abs().max()), float(want.abs().max())
        assert got.shape == want.shape and err <= tol * scale, (what, err, scale)


@pytest.mark.parametrize("create_graph", [False, True])
def test_weight_changed_before_the_backward_pass(create_graph):
    """As under stock autocast, which keeps the rounded copy: the gradients are those of the weight of the forward pass."""
    print(f"linear, weight changed in place, create_graph={create_graph}", flush=True)
    g = torch.Generator().manual_seed(4)
    x, w = torch.randn(2, 600, 64, generator=g).bfloat16().cuda().requires_grad_(True), torch.randn(72, 64, generator=g).cuda().requires_grad_(True)
    grad = torch.randn(2, 600, 72, generator=g).bfloat16().cuda()
    got = []
    for f in (lambda: hip_backend().linear(x, w), lambda: torch.nn.functional.linear(x, w)):
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = f()
        with torch.no_grad():
            w.mul_(2)
        got.append(torch.autograd.grad(y, (x, w), grad, create_graph=create_graph))
        with torch.no_grad():
            w.div_(2)
    for (a, b), tol in zip(zip(*got), (1e-6, ULP[torch.bfloat16])):   # the same product; the stock gradient of w is rounded to bf16
        a, b = a.detach(), b.detach()
        assert a.dtype == b.dtype and float((a.float() - b.float()).abs().max()) <= tol * float(b.float().abs().max())


def test_gradient_of_a_gradient():
    """Second derivatives against fp64 products of the rounded operands: a handful of bf16 roundings."""
    print("linear, second derivative", flush=True)
    g = torch.Generator().manual_seed(5)
    x, w = torch.randn(1100, 64, generator=g).bfloat16().cuda().requires_grad_(True), (torch.randn(72, 64, generator=g) / 8).bfloat16().float().cuda().requires_grad_(True)
    wide = [t.detach().double().requires_grad_(True) for t in (x, w)]
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = hip_backend().linear(x, w)
    results = []
    for out, leaves in ((y, (x, w)), (wide[0] @ wide[1].T, wide)):
        first = torch.autograd.grad(out.float().square().sum() if out is y else out.square().sum(), leaves, create_graph=True)
        results.append(torch.autograd.grad(sum(t.to(out.dtype if out is not y else torch.float32).square().sum() for t in first), leaves))
    for got, want in zip(*results):
        assert float((got.double() - want).abs().max()) <= 2.0 ** -6 * float(want.abs().max())


def test_other_calls_stay_stock():
    x = torch.randn(2, 1024, 64, device="cuda", dtype=torch.bfloat16)
    w = torch.randn(64, 64, device="cuda", requires_grad=True)
    assert not dense.is_linear_supported(x, w)   # without autocast the types do not go together
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert dense.is_linear_supported(x, w)
        assert not dense.is_linear_supported(x[:, :8], w) and not dense.is_linear_supported(x, w.detach()) and not dense.is_linear_supported(x.float(), w)
        with torch.no_grad():
            assert not dense.is_linear_supported(x, w)
    with torch.autocast("cuda", dtype=torch.float16):
        assert not dense.is_linear_supported(x, w)


@pytest.mark.parametrize("T,N,K", [(1, 64, 64), (2, 2304, 768), (127, 320, 256), (128, 128, 320), (129, 1000, 264), (1500, 2304, 768), (1792, 2304, 768), (8191, 768, 768),
                                   (300, 16384, 128), (22100, 776, 512)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_products(T, N, K, dtype):
    """The products alone: a row, tiles and one row more or less, a round of small tiles and its last, rounds of large ones, sums of whole k-tiles and others."""
    from minitrain_amd import _lib

    print(f"linear products T={T} N={N} K={K} {dtype}", flush=True)
    lib, act, stream = _lib.load(), _lib.dtype_code(dtype), torch.cuda.current_stream().cuda_stream
    g = torch.Generator().manual_seed(T + N)
    x, w, grad = (torch.randn(*s, generator=g).to(dtype).cuda() for s in ((T, K), (N, K), (T, N)))
    y, dx = torch.full((T, N), float("nan"), dtype=dtype, device="cuda"), torch.full((T, K), float("nan"), dtype=dtype, device="cuda")
    _lib.check(lib.mts_linear_fwd(x.data_ptr(), w.data_ptr(), T, N, K, act, y.data_ptr(), stream), "mts_linear_fwd")
    _lib.check(lib.mts_linear_dx(grad.data_ptr(), w.data_ptr(), T, N, K, act, dx.data_ptr(), stream), "mts_linear_dx")
    for got, want in ((y, x.double() @ w.double().T), (dx, grad.double() @ w.double())):
        assert float((got.double() - want).abs().max()) <= ULP[dtype] * float(want.abs().max())


@pytest.mark.parametrize("T,N,K", [(16, 768, 768), (1000, 2304, 768), (300, 1000, 264)])
def test_projection_without_gradients(T, N, K):
    """Evaluation under autocast: the product that the stock operator gives, its cached rounding of the weight, and no graph."""
    g = torch.Generator().manual_seed(T)
    x, w = torch.randn(1, T, K, generator=g).bfloat16().cuda(), torch.randn(N, K, generator=g).cuda().requires_grad_(True)
    ops = hip_backend()
    for context in (torch.no_grad, torch.inference_mode):
        with context(), torch.autocast("cuda", dtype=torch.bfloat16):
            y, stock = ops.linear(x, w), torch.nn.functional.linear(x, w)
            w_before = w.detach().clone()
            if context is torch.no_grad:   # a weight changed inside the context: autocast goes on with its copy
                w.mul_(2)
                assert torch.equal(ops.linear(x, w), y) and torch.equal(torch.nn.functional.linear(x, w), stock)
                w.copy_(w_before)
        assert not y.requires_grad and y.shape == (1, T, N)
        want = x.double() @ w.detach().bfloat16().double().T
        assert float((y.double() - want).abs().max()) <= ULP[torch.bfloat16] * float(want.abs().max())
    with torch.no_grad():
        assert ops.linear(x, w) is None   # no autocast
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert ops.linear(x[..., 1:], w[:, 1:]) is None and ops.linear(x.transpose(1, 2), torch.zeros(8, T, device="cuda")) is None
