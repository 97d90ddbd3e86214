"""The layer's forward pass for few tokens in two launches, against the entry points that it stands for (GPU).

Logits are fp32 sums of H products in another order: within 2^-20 of the sum of the products' sizes.  Everything behind them is the same arithmetic on the
same values: routing and rows exactly, the expert rows and the output to the bit when the other entry points are given its routing weights."""

import pytest
import torch

from minitrain_amd import _lib
from oracle import moe_oracle as O
from tests.helpers import BF16_TOL, assert_close_scaled, hip_backend
from tests.test_gpu_layer_node import _layer_grads

pytestmark = pytest.mark.gpu


def _run(lib, x, w_r, w1, w2, K, normalize, with_pre):
    T, H = x.shape
    E, I, TK = w_r.shape[0], w1.shape[1] // 2, T * K
    act, wcode = _lib.dtype_code(x.dtype), _lib.dtype_code(w1.dtype)
    assert lib.mts_moe_few_tokens_supported(act, wcode, T, K, E, H, I)
    f = lambda *s: torch.full(s, float("nan"), device="cuda")
    i = lambda n: torch.full((n,), -7, dtype=torch.int32, device="cuda")
    a = lambda *s: torch.full(s, float("nan"), dtype=x.dtype, device="cuda")
    o = dict(logits=f(T, E), weights=f(T, K), indices=i(TK).view(T, K), weights_act=a(T, K), prob=f(E), z=f(1), entropy=f(1), counts=i(E), lb=f(1), load=f(E + 7),
             start=i(E + 1), scatter=i(TK), reverse=i(TK), gather=i(TK), pre=a(TK, 2 * I) if with_pre else None, post=a(TK, I), y=a(TK, H),
             arrived=i((H + 31) // 32), out=a(T, H))
    p = lambda t: None if t is None else t.data_ptr()
    _lib.check(lib.mts_moe_few_tokens_fwd(p(x), p(w_r), p(w1), p(w2), wcode, T, H, E, I, K, int(normalize), act, *(p(t) for t in o.values()),
                                          torch.cuda.current_stream().cuda_stream), "mts_moe_few_tokens_fwd")
    return o


@pytest.mark.parametrize("T,K,E,H,I", [
    (1, 1, 1, 8, 8), (1, 2, 8, 768, 1024), (2, 2, 8, 64, 40), (3, 4, 9, 72, 96), (15, 2, 8, 776, 264), (16, 2, 8, 768, 1024), (17, 2, 8, 768, 1000),
    (16, 8, 16, 256, 72), (31, 3, 12, 1024, 512), (32, 8, 8, 200, 1368), (32, 1, 16, 2048, 136), (9, 5, 5, 4096, 64), (5, 2, 3, 16, 32)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("masters", [False, True])
def test_few_tokens(T, K, E, H, I, dtype, masters):
    """One token to two full tiles, one to sixteen experts, all of them chosen and most of them idle, widths that are not whole tiles."""
    print(f"few tokens T={T} K={K} E={E} H={H} I={I} {dtype} masters={masters}", flush=True)
    lib = _lib.load()
    if masters and E > 8:
        assert not lib.mts_moe_few_tokens_supported(_lib.dtype_code(dtype), _lib.dtype_code(torch.float32), T, K, E, H, I)
        return
    x, w_r, w1, w2, _ = O.make_inputs(900 + T + E, T, H, E, I)
    x, w_r = x.to(dtype).cuda(), w_r.cuda()
    w1, w2 = (t.to(torch.float32 if masters else dtype).cuda() for t in (w1, w2))
    normalize = T % 2 == 0
    o = _run(lib, x, w_r, w1, w2, K, normalize, True)
    TK, act, stream = T * K, _lib.dtype_code(dtype), torch.cuda.current_stream().cuda_stream
    # logits in fp64
    xd, wd = x.double(), w_r.double()
    assert bool(((o["logits"].double() - xd @ wd.T).abs() <= 2.0 ** -20 * (xd.abs() @ wd.abs().T)).all())
    # post-process of these logits
    ref = O.router_postprocess(o["logits"].cpu(), K, normalize=normalize)
    assert torch.equal(o["indices"].cpu(), ref.expert_indices)
    torch.testing.assert_close(o["weights"].cpu(), ref.expert_weights, rtol=2e-5, atol=1e-7)
    assert torch.equal(o["weights_act"], o["weights"].to(dtype))
    for name, want in (("prob", ref.probability_per_expert), ("z", ref.z_loss), ("entropy", ref.entropy)):
        torch.testing.assert_close(o[name].cpu().view(want.shape), want, rtol=2e-5, atol=1e-6)
    counts, start, scatter, reverse, gather = (torch.empty(n, dtype=torch.int32, device="cuda") for n in (E, E + 1, TK, TK, TK))
    n = lib.mts_moe_route_workspace_bytes(T, K, E)
    ws = torch.empty(max(n, 4), dtype=torch.uint8, device="cuda")
    _lib.check(lib.mts_moe_route(o["indices"].data_ptr(), T, K, E, 64, counts.data_ptr(), start.data_ptr(), scatter.data_ptr(), reverse.data_ptr(),
                                 gather.data_ptr(), None, None, None, ws.data_ptr(), n, stream), "mts_moe_route")
    for name, want in (("counts", counts), ("start", start), ("scatter", scatter), ("reverse", reverse), ("gather", gather)):
        assert torch.equal(o[name], want), name
    share = counts.cpu().double() / TK
    torch.testing.assert_close(o["lb"].cpu().double()[0], E * (share * ref.probability_per_expert.double()).sum(), rtol=2e-5, atol=1e-6)
    torch.testing.assert_close(o["load"].cpu().double()[:E], share, rtol=1e-6, atol=0)
    # the experts with these routing weights
    pre, post, y, out = (torch.empty_like(t) for t in (o["pre"], o["post"], o["y"], o["out"]))
    _lib.check(lib.mts_moe_fwd_few_rows(x.data_ptr(), w1.data_ptr(), w2.data_ptr(), _lib.dtype_code(w1.dtype), gather.data_ptr(), start.data_ptr(),
                                        o["weights_act"].data_ptr(), scatter.data_ptr(), T, K, E, H, I, act, pre.data_ptr(), post.data_ptr(), y.data_ptr(), stream),
               "mts_moe_fwd_few_rows")
    _lib.check(lib.mts_moe_combine(y.data_ptr(), None, None, reverse.data_ptr(), T, K, H, act, out.data_ptr(), stream), "mts_moe_combine")
    for name, want in (("pre", pre), ("post", post), ("y", y), ("out", out)):
        assert torch.equal(o[name], want), name
    again = _run(lib, x, w_r, w1, w2, K, normalize, False)   # pre-activations that nobody wants, and the same to the bit
    assert all(torch.equal(again[name], o[name]) for name in o if name != "pre")


def test_few_tokens_of_ties_and_of_no_number():
    """Equal logits go to the lower experts, also across the blocks that work the routing out each for itself; a row that is no number has
    experts of its own and leaves the others' results alone."""
    lib = _lib.load()
    T, K, E, H, I = 20, 2, 8, 128, 64
    x, w_r, w1, w2, _ = (t.cuda() for t in O.make_inputs(31, T, H, E, I))
    x, w1, w2 = x.bfloat16(), w1.bfloat16(), w2.bfloat16()
    w_r[5] = w_r[1]
    x[3] = 0
    clean = _run(lib, x, w_r, w1, w2, K, True, True)
    assert clean["indices"][3].tolist() == [0, 1]
    chosen = torch.zeros(T, E, dtype=torch.bool).scatter_(1, clean["indices"].cpu().long(), True)
    assert bool((~chosen[:, 5] | chosen[:, 1]).all())
    x[7] = float("nan")
    o = _run(lib, x, w_r, w1, w2, K, True, True)
    assert len(set(o["indices"][7].tolist())) == K and bool(o["out"][7].isnan().all())
    others = [t for t in range(T) if t != 7]
    assert torch.equal(o["out"][others], clean["out"][others]) and torch.equal(o["indices"][others], clean["indices"][others])


@pytest.mark.parametrize("T,K,E,H,I", [(2, 2, 8, 768, 1024), (5, 1, 4, 64, 40), (16, 2, 8, 256, 128), (17, 2, 8, 776, 264), (31, 4, 8, 128, 512), (32, 2, 16, 512, 256)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("masters", [False, True])
def test_layer_of_few_tokens_and_its_gradients(T, K, E, H, I, dtype, masters):
    """The layer node, which takes the two launches, against the oracle in fp32 on the same rounded values."""
    print(f"layer of few tokens T={T} K={K} E={E} H={H} I={I} {dtype} masters={masters}", flush=True)
    act = _lib.dtype_code(dtype)
    assert _lib.load().mts_moe_few_tokens_preferred(act, act, T, K, E, H, I)   # a backward pass follows: the weights are rounded first
    x, w_r, w1, w2, g = O.make_inputs(70 + T, T, H, E, I)
    res, grads = _layer_grads(hip_backend(), dict(x=x, w_r=w_r, w1=w1, w2=w2, g=g), K, True, dtype, masters)
    kept = torch.float32 if masters else dtype
    leaves = [x.to(dtype).float().requires_grad_(True), w_r.clone().requires_grad_(True), w1.to(kept).float().requires_grad_(True), w2.to(kept).float().requires_grad_(True)]
    hidden, r = O.moe_feed_forward(leaves[0].to(dtype), leaves[1], leaves[2].to(kept), leaves[3].to(kept), K, normalize=True, compute_dtype=torch.float32)
    ((hidden * g.to(dtype).float()).sum() + 0.01 * r.auxiliary_loss + 0.001 * r.z_loss).backward()
    assert torch.equal(res[7].cpu(), r.expert_indices)
    assert_close_scaled(res[0], hidden, BF16_TOL, "hidden")
    torch.testing.assert_close(res[1].cpu(), r.auxiliary_loss, rtol=1e-4, atol=1e-6)
    torch.testing.assert_close(res[2].cpu(), r.z_loss, rtol=1e-4, atol=1e-6)
    for name, got, leaf in zip(("dx", "dW_r", "dW1", "dW2"), grads, leaves):
        assert_close_scaled(got, leaf.grad, BF16_TOL, name)


@pytest.mark.parametrize("T,masters", [(1, False), (16, False), (32, True)])
def test_few_tokens_in_a_graph_and_on_two_streams(T, masters):
    """Replays of a graph with other tokens and eager calls between them, and calls on two streams at a time, each with its own tokens: the counters of
    the second launch are a call's own and cleared by its first, so all give what calls one after the other give."""
    print(f"few tokens in a graph and on two streams T={T} masters={masters}", flush=True)
    ops, K, E, H, I = hip_backend(), 2, 8, 768, 1024
    _, w_r, w1, w2, _ = (t.cuda() for t in O.make_inputs(5, T, H, E, I))
    if not masters:
        w1, w2 = w1.bfloat16(), w2.bfloat16()
    g = torch.Generator().manual_seed(4)
    tokens = [torch.randn(T, H, generator=g).bfloat16().cuda() for _ in range(8)]
    with torch.no_grad():
        want = [ops.moe_layer(x, w_r, w1, w2, K, normalize=True)[0].clone() for x in tokens]
        x = tokens[0].clone()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = ops.moe_layer(x, w_r, w1, w2, K, normalize=True)[0]
        for t, w in zip(tokens, want):
            x.copy_(t)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, w)
            assert torch.equal(ops.moe_layer(t, w_r, w1, w2, K, normalize=True)[0], w)
        streams = [torch.cuda.Stream() for _ in range(2)]
        for s in streams:
            s.wait_stream(torch.cuda.current_stream())
        got = {}
        for repeat in range(10):
            for i, t in enumerate(tokens):
                with torch.cuda.stream(streams[i % 2]):
                    got[repeat, i] = ops.moe_layer(t, w_r, w1, w2, K, normalize=True)[0]
        torch.cuda.synchronize()
        assert all(torch.equal(o, want[i]) for (_, i), o in got.items())
