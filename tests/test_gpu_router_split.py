"""The router projection of more than 16 experts and its gradients for bf16 rows: fp32 operands as three bf16 terms (GPU).

Every value of those operands is the sum of its terms and every product exact, so that what is left is the rounding of fp32 sums: within 2^-20 of the sum of
the products' sizes, as for the fp32 instruction; dx is rounded to bf16 once more."""

import pytest
import torch

from minitrain_amd import _lib

pytestmark = pytest.mark.gpu


def _forward(lib, x, w):
    logits = torch.full((x.shape[0], w.shape[0]), float("nan"), device="cuda")
    _lib.check(lib.mts_router_wide_fwd(x.data_ptr(), w.data_ptr(), *x.shape, w.shape[0], _lib.dtype_code(x.dtype), logits.data_ptr(),
                                       torch.cuda.current_stream().cuda_stream), "mts_router_wide_fwd")
    return logits


def _backward(lib, dl, x, w):
    dx, dw = torch.full_like(x, float("nan")), torch.full_like(w, float("nan"))
    size = lib.mts_router_wide_bwd_workspace_bytes(*x.shape, w.shape[0])
    ws = torch.empty(size, dtype=torch.uint8, device="cuda")
    _lib.check(lib.mts_router_wide_bwd(dl.data_ptr(), x.data_ptr(), w.data_ptr(), *x.shape, w.shape[0], _lib.dtype_code(x.dtype), dx.data_ptr(), dw.data_ptr(),
                                       ws.data_ptr(), size, torch.cuda.current_stream().cuda_stream), "mts_router_wide_bwd")
    return dx, dw


def _check(got, a, b, extra=0.0):
    """got against a @ b in fp64"""
    a, b = a.double(), b.double()
    want = a @ b
    assert bool(((got.double() - want).abs() <= 2.0 ** -20 * (a.abs() @ b.abs()) + extra * want.abs()).all())


@pytest.mark.parametrize("E", [17, 24, 32, 40, 64, 72, 128, 136])
@pytest.mark.parametrize("T,H", [(65, 136), (1023, 64), (1024, 8), (1025, 72), (1153, 768), (2050, 1032), (4099, 200)])
def test_router_split(T, H, E):
    """Rows, columns and experts around whole tiles and steps; experts that are no whole eights and more of them than the terms' tile holds."""
    print(f"router split T={T} H={H} E={E}", flush=True)
    lib = _lib.load()
    g = torch.Generator().manual_seed(T + H + E)
    x, w = torch.randn(T, H, generator=g).bfloat16().cuda(), (torch.randn(E, H, generator=g) * 0.05).cuda()
    dl = (torch.randn(T, E, generator=g) * 1e-4).cuda()
    dl[T // 2] = 0   # a row without a gradient
    _check(_forward(lib, x, w), x, w.T)
    dx, dw = _backward(lib, dl, x, w)
    _check(dx, dl, w, 2.0 ** -8)
    _check(dw, dl.T, x)
    again = _backward(lib, dl, x, w)
    assert torch.equal(again[0], dx) and torch.equal(again[1], dw)


@pytest.mark.parametrize("where", ["x", "w", "dl"])
@pytest.mark.parametrize("value", [float("inf"), float("nan"), 3e38, 2.0 ** -100, 2.0 ** 60])
@pytest.mark.parametrize("T,H,E", [(1100, 264, 64), (1025, 72, 24), (1041, 72, 128)])
def test_router_split_of_values_that_do_not_split(T, H, E, where, value):
    """Infinities, NaN, and values whose terms would leave the range, alone among ordinary ones: the sums that hold them are what fp32 sums give, the
    others stay what they are."""
    print(f"router split T={T} H={H} E={E} {where}={value}", flush=True)
    lib = _lib.load()
    g = torch.Generator().manual_seed(9)
    t = dict(x=torch.randn(T, H, generator=g).bfloat16(), w=torch.randn(E, H, generator=g) * 0.05, dl=torch.randn(T, E, generator=g) * 1e-4)
    row, col = t[where].shape[0] - 3, t[where].shape[1] - 2
    clean = {k: v.cuda() for k, v in t.items()}
    t[where][row, col] = value
    t = {k: v.cuda() for k, v in t.items()}
    dx0, dw0 = _backward(lib, clean["dl"], clean["x"], clean["w"])
    y0 = _forward(lib, clean["x"], clean["w"])
    y, (dx, dw) = _forward(lib, t["x"], t["w"]), _backward(lib, t["dl"], t["x"], t["w"])
    for name, got, base, a, b, extra in (("y", y, y0, "x", "wT", 0.0), ("dx", dx, dx0, "dl", "w", 2.0 ** -8), ("dw", dw, dw0, "dlT", "x", 0.0)):
        operand = lambda n: t[n[:-1]].T if n.endswith("T") else t[n]
        a, b = operand(a).double(), operand(b).double()
        want = a @ b
        finite = want.abs() < 3e38
        over = (want.abs() > 3.5e38) & want.isfinite()
        bound = 2.0 ** -20 * (a.abs() @ b.abs()) + extra * want.abs()
        assert bool(((got.double() - want).abs() <= bound)[finite].all()), name
        assert torch.equal(got.isnan(), want.isnan()), name
        assert bool((got.double() == want)[want.isinf()].all()) and bool((got.isinf() | (got.abs() > 3e38))[over].all()), name


def _confident(T, E, std, g):
    """dlogits as a router leaves them whose logits have this spread: p * (something of its own)"""
    p = torch.softmax(torch.randn(T, E, generator=g).cuda() * std, dim=-1)
    return (p * torch.randn(T, E, generator=g).cuda() * 1e-4).contiguous()


@pytest.mark.parametrize("std", [5, 12, 40])
@pytest.mark.parametrize("T,H,E", [(1024, 264, 64), (1041, 72, 24), (2050, 136, 128), (1300, 520, 32)])
def test_router_split_of_confident_routers(T, H, E, std):
    """dlogits over the whole range of fp32, down to zeros.  Beside the bound of the sums: up to 2^10 roundings to a multiple of the
    smallest number, 2^-149, in dw."""
    print(f"router split T={T} H={H} E={E} std={std}", flush=True)
    lib = _lib.load()
    g = torch.Generator().manual_seed(T + std)
    x, w, dl = torch.randn(T, H, generator=g).bfloat16().cuda(), (torch.randn(E, H, generator=g) * 0.05).cuda(), _confident(T, E, std, g)
    dl[:, 3] *= 2.0 ** -90   # an expert that hardly any token hears of
    dx, dw = _backward(lib, dl, x, w)
    _check(dx, dl, w, 2.0 ** -8)
    want, sizes = dl.double().T @ x.double(), dl.double().abs().T @ x.double().abs()
    assert bool(((dw.double() - want).abs() <= 2.0 ** -20 * sizes + 2.0 ** -139).all())


@pytest.mark.parametrize("where,border", [("x", 2.0 ** 40), ("w", 2.0 ** 16), ("dl", 2.0 ** 36)])
@pytest.mark.parametrize("below", [True, False])
def test_router_split_up_to_the_largest_values_that_it_takes(where, border, below):
    """Operands that are as large as the split takes them throughout, and one value beyond."""
    lib = _lib.load()
    g = torch.Generator().manual_seed(11)
    T, H, E = 1041, 136, 64
    t = dict(x=torch.rand(T, H, generator=g) - 0.5, w=torch.rand(E, H, generator=g) - 0.5, dl=torch.rand(T, E, generator=g) - 0.5)
    t[where] *= 2 * border * (1 - 2.0 ** -8)
    if not below:
        t[where][t[where].shape[0] // 2, 5] = border
    x, w, dl = t["x"].bfloat16().cuda(), t["w"].cuda(), t["dl"].cuda()
    dx, dw = _backward(lib, dl, x, w)
    _check(dx, dl, w, 2.0 ** -8)
    _check(dw, dl.T, x)


@pytest.mark.parametrize("T,H,E", [(8192, 1024, 64), (16384, 2048, 128)])
def test_router_split_is_as_fast_for_small_and_large_gradients(T, H, E):
    """The split takes values of all sizes below its border, those of confident routers and of a loss that is scaled among them: the same work for any dlogits,
    and a quarter of its time for noise."""
    lib = _lib.load()
    g = torch.Generator().manual_seed(3)
    x, w = torch.randn(T, H, generator=g).bfloat16().cuda(), (torch.randn(E, H, generator=g) * 0.05).cuda()

    def time_of(dl):
        times = []
        for _ in range(7):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            for _ in range(10):
                _backward(lib, dl, x, w)
            end.record()
            torch.cuda.synchronize()
            times.append(start.elapsed_time(end))
        return min(times)

    ordinary = _confident(T, E, 1, g)
    time_of(ordinary)
    for other in (_confident(T, E, 12, g), 2.0 ** 40 * ordinary):
        assert time_of(other) <= 1.25 * time_of(ordinary)
