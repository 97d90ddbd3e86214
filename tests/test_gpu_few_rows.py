"""Expert GEMMs for few rows per expert, against the same products in fp64 and next to the general kernels (GPU).

Tolerance, relative to the largest value: one rounding of a result to the 16-bit type (2^-9, 2^-12) and, where rounded values
enter the next product, one more: 2^-8 and 2^-11 for the pre-activation, twice that for the others."""

import pytest
import torch

from minitrain_amd import _lib
from minitrain_amd.kernels.hip.fused_moe import routing_for_experts
from minitrain_amd.kernels.hip.moe_layer import moe_layer
from minitrain_amd.model.ops import get_ops_backend

pytestmark = pytest.mark.gpu

ULP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _close(got, want, tol, what):
    err, scale = float((got.double() - want).abs().max()), float(want.abs().max())
    assert err <= tol * scale, (what, err, scale)


@pytest.mark.parametrize("T,K,E,H,I", [
    (1, 1, 1, 8, 8), (3, 2, 4, 64, 32), (16, 2, 8, 768, 1024), (33, 1, 2, 72, 40), (17, 1, 1, 192, 264), (65, 1, 1, 1000, 136),
    (40, 4, 70, 256, 96), (129, 2, 5, 320, 1368), (200, 1, 3, 2056, 24)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("weight_dtype", ["same", "fp32"])
@pytest.mark.parametrize("weighted", [True, False])
def test_few_rows(T, K, E, H, I, dtype, weight_dtype, weighted):
    """One row to full tiles of 16, 32 and 64 and one more, experts without rows, more experts than a wave has lanes, columns
    and k that are not whole tiles or steps, routes that were dropped."""
    print(f"few rows T={T} K={K} E={E} H={H} I={I} {dtype} weights {weight_dtype} weighted={weighted}", flush=True)
    lib = _lib.load()
    g = torch.Generator().manual_seed(T + H)
    wt = torch.float32 if weight_dtype == "fp32" else dtype
    x = torch.randn(T, H, generator=g).to(dtype).cuda()
    w1 = (torch.randn(E, 2 * I, H, generator=g) * H ** -0.5).to(wt).cuda()
    w2 = (torch.randn(E, H, I, generator=g) * I ** -0.5).to(wt).cuda()
    idx = torch.stack([torch.randperm(E, generator=g)[:K] for _ in range(T)]).int().cuda()
    if T > 16:
        idx[T // 2, 0] = -1   # a dropped route
    weights = torch.rand(T, K, generator=g).to(dtype).cuda()
    start, gather, scatter, _ = routing_for_experts(idx, E)
    rows = int(start[E])
    TK = T * K
    act, wcode = _lib.dtype_code(dtype), _lib.dtype_code(wt)
    assert lib.mts_moe_fwd_few_rows_supported(act, wcode, T, TK, E, H, I)
    out = lambda width: torch.full((TK, width), float("nan"), dtype=dtype, device="cuda")
    pre, post, y = out(2 * I), out(I), out(H)
    route_w, route_e = (weights.data_ptr(), scatter.data_ptr()) if weighted else (None, None)
    stream = torch.cuda.current_stream().cuda_stream
    _lib.check(lib.mts_moe_fwd_few_rows(x.data_ptr(), w1.data_ptr(), w2.data_ptr(), wcode, gather.data_ptr(), start.data_ptr(), route_w, route_e, T, K, E, H, I,
                                        act, pre.data_ptr(), post.data_ptr(), y.data_ptr(), stream), "mts_moe_fwd_few_rows")
    n1, n2 = w1.to(dtype), w2.to(dtype)   # the weights enter the products rounded, on either path
    pre2, post2, y2 = out(2 * I), out(I), out(H)
    _lib.check(lib.mts_moe_fwd_gateup_swiglu(x.data_ptr(), n1.data_ptr(), gather.data_ptr(), start.data_ptr(), route_w, route_e, T, K, E, H, I, act,
                                             pre2.data_ptr(), post2.data_ptr(), stream), "mts_moe_fwd_gateup_swiglu")
    _lib.check(lib.mts_moe_fwd_down(post2.data_ptr(), n2.data_ptr(), start.data_ptr(), TK, E, H, I, act, y2.data_ptr(), stream), "mts_moe_fwd_down")
    bounds = start.tolist()
    for e in range(E):
        a, b = bounds[e], bounds[e + 1]
        if a == b:
            continue
        want = x[gather[a:b].long()].double() @ n1[e].double().T
        gate, up = want[:, :I], want[:, I:]
        s = weights.view(-1)[scatter[a:b].long()].double()[:, None] if weighted else 1.0
        act_want = torch.nn.functional.silu(gate) * up * s
        _close(pre[a:b], want, ULP[dtype], "pre")
        _close(post[a:b], act_want, 2 * ULP[dtype], "post")
        _close(y[a:b], post[a:b].double() @ n2[e].double().T, ULP[dtype], "y")
    for got, other, what in ((pre, pre2, "pre"), (post, post2, "post"), (y, y2, "y")):
        _close(got[:rows], other[:rows].double(), 2 * ULP[dtype], f"{what} next to the general kernels")
        assert got[rows:].isnan().all()   # rows behind the last expert's are left alone


@pytest.mark.parametrize("T", [24, 700, 20000])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_layer_with_and_without_a_backward_pass(T, dtype):
    """Where no backward pass follows the pre-activations are not kept and few rows read fp32 weights as they are: the same result
    as with one, for few rows, small tiles and the joint launch."""
    print(f"layer, master weights, T={T} {dtype}", flush=True)
    g = torch.Generator().manual_seed(2)
    x = torch.randn(T, 256, generator=g).to(dtype).cuda()
    w_r, w1, w2 = ((torch.randn(*s, generator=g) * 0.05).cuda().requires_grad_(True) for s in ((8, 256), (8, 512, 256), (8, 256, 256)))
    trained = moe_layer(x, w_r, w1, w2, 2, normalize=True)[0]
    with torch.no_grad():
        read = moe_layer(x, w_r, w1, w2, 2, normalize=True)[0]
    assert torch.equal(trained, read)
    trained.sum().backward()
    assert all(t.grad.isfinite().all() for t in (w_r, w1, w2))


@pytest.mark.parametrize("T,K,E,H,I", [(64, 2, 8, 768, 1024), (65, 2, 8, 768, 1024), (65, 1, 8, 512, 512), (193, 1, 8, 1024, 512), (96, 2, 8, 512, 2048), (97, 2, 8, 512, 2048),
                                       (192, 2, 8, 1024, 2048), (193, 2, 8, 1024, 2048), (64, 2, 16, 768, 1024), (65, 2, 16, 768, 1024)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_either_side_of_the_rule(T, K, E, H, I, dtype):
    """fp32 master weights without a backward pass, read as they are or rounded first, on both sides of every line of the rule: as with weights that were rounded
    before.  The two sum the same products in other orders, which moves a rounding of either expert row or of the output by one step at most."""
    print(f"few rows rule T={T} K={K} E={E} H={H} I={I} {dtype}", flush=True)
    g = torch.Generator().manual_seed(T + H)
    x = torch.randn(T, H, generator=g).to(dtype).cuda()
    w_r = torch.randn(E, H, generator=g).cuda()
    w1, w2 = (torch.randn(E, 2 * I, H, generator=g) * H ** -0.5).cuda(), (torch.randn(E, H, I, generator=g) * I ** -0.5).cuda()
    with torch.no_grad():
        got, want = (moe_layer(x, w_r, a, b, K, normalize=True)[0] for a, b in ((w1, w2), (w1.to(dtype), w2.to(dtype))))
    _close(got, want.double(), 4 * ULP[dtype], "out")


@pytest.mark.parametrize("call", ["operator", "layer"])
def test_masters_of_many_experts_are_not_copied(call):
    """Without a backward pass: no rounded copies of 75 M weights for 9 rows an expert, where they would be a launch of their own (the operator, and a layer of
    more experts than the head's launches carry copies for)."""
    T, K, E, H, I = 300, 4, 128, 768, 256
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randn(T, H, generator=g, device="cuda").bfloat16()
    w1, w2 = torch.randn(E, 2 * I, H, generator=g, device="cuda") * H ** -0.5, torch.randn(E, H, I, generator=g, device="cuda") * I ** -0.5
    w_r = torch.randn(E, H, generator=g, device="cuda")
    ops = get_ops_backend("hip")

    def run(a, b):
        if call == "layer":
            return moe_layer(x, w_r, a, b, K, normalize=True)[0]
        route = ops.router_postprocess(x.float() @ w_r.T, K, normalize=True)
        return ops.fused_moe(x, a, b, route.expert_indices, route.expert_weights.bfloat16())

    with torch.no_grad():
        want = run(w1.bfloat16(), w2.bfloat16())
        before = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        got = run(w1, w2)
    assert torch.cuda.max_memory_allocated() - before < w1.numel()   # the copies: three bytes for each of these
    _close(got, want.double(), 4 * ULP[torch.bfloat16], "out")
