"""The chained head of 17 to 64 experts against the separate operators and the oracle."""

import pytest
import torch

from oracle import moe_oracle as O

pytestmark = pytest.mark.gpu


def _head(x, w_r, K, normalize):
    from minitrain_amd import _lib

    lib = _lib.load()
    (T, H), E = x.shape, w_r.shape[0]
    f32, i32 = dict(dtype=torch.float32, device="cuda"), dict(dtype=torch.int32, device="cuda")
    o = dict(logits=torch.empty(T, E, **f32), weights=torch.empty(T, K, **f32), indices=torch.empty(T, K, **i32),
             weights_act=torch.empty(T, K, dtype=x.dtype, device="cuda") if x.dtype != torch.float32 else None,
             prob_mean=torch.empty(E, **f32), z_loss=torch.empty(1, **f32), entropy=torch.empty(1, **f32), counts=torch.empty(E, **i32),
             load_balance=torch.empty(1, **f32), load_stats=torch.empty(E + 7, **f32), expert_start=torch.empty(E + 1, **i32),
             s_scatter=torch.full((T * K,), -9, **i32), s_reverse=torch.full((T * K,), -9, **i32), x_gather=torch.full((T * K,), -9, **i32))
    size = lib.mts_moe_wide_head_workspace_bytes(T, E)
    ws = torch.empty(size, dtype=torch.uint8, device="cuda")
    call = lambda bytes: lib.mts_moe_wide_head_fwd(x.data_ptr(), w_r.data_ptr(), T, H, E, K, int(normalize), _lib.dtype_code(x.dtype),
                                                   *[_lib.ptr(t) for t in o.values()], ws.data_ptr(), bytes, _lib.stream_of(x))
    assert call(size - 4) == -4   # refused on the host
    assert call(size) == 0
    return o


@pytest.mark.parametrize("T,H,E,K,dtype,normalize", [
    (1, 4, 17, 1, torch.float32, True), (31, 64, 24, 8, torch.float16, True), (33, 60, 32, 2, torch.bfloat16, False), (257, 768, 33, 4, torch.bfloat16, True),
    (600, 1024, 64, 4, torch.bfloat16, True), (1000, 132, 63, 3, torch.float32, False), (8191, 200, 48, 8, torch.float16, True), (32768, 64, 64, 2, torch.bfloat16, True)])
def test_chained_head_equals_the_separate_operators(T, H, E, K, dtype, normalize):
    print(f"wide head T={T} H={H} E={E} K={K} {dtype} normalize={normalize}", flush=True)
    from minitrain_amd.kernels.hip.fused_moe import compute_routing_metadata
    from minitrain_amd.kernels.hip.router import router_logits, router_postprocess

    x, w_r, _, _, _ = O.make_inputs(T + E, T, H, E, 8)
    x, w_r = x.to(dtype).cuda(), w_r.cuda()
    x[::7] = 0   # ties of all experts: the lowest indices
    w_r[E // 2] = w_r[1]
    got = _head(x, w_r, K, normalize)
    logits = router_logits(x, w_r)
    route = router_postprocess(logits, K, normalize=normalize, weights_dtype=None if dtype == torch.float32 else dtype)
    assert torch.equal(got["logits"], logits) and torch.equal(got["indices"], route.expert_indices) and torch.equal(got["counts"], route.expert_counts)
    assert torch.equal(got["weights"], route.expert_weights)   # the same lanes a row
    assert dtype == torch.float32 or torch.equal(got["weights_act"], got["weights"].to(dtype))
    assert torch.equal(got["indices"][::7].cpu(), torch.arange(K, dtype=torch.int32).expand(len(range(0, T, 7)), K))
    for name, want in (("prob_mean", route.probability_per_expert), ("z_loss", route.z_loss), ("entropy", route.entropy), ("load_balance", route.load_balance_loss),
                       ("load_stats", route.load_stats)):   # sums over blocks of other sizes
        torch.testing.assert_close(got[name].flatten(), want.flatten(), rtol=2e-5, atol=2e-6, msg=name)
    assert torch.equal(got["indices"].cpu(), O.router_postprocess(logits.cpu(), K, normalize=normalize).expert_indices)
    counts, start, gather, scatter, reverse, *_ = compute_routing_metadata(got["indices"], E)
    assert torch.equal(got["counts"], counts) and torch.equal(got["expert_start"], start)
    assert torch.equal(got["s_scatter"], scatter) and torch.equal(got["s_reverse"], reverse) and torch.equal(got["x_gather"], gather)


def test_what_the_chain_does_not_take():
    from minitrain_amd import _lib

    takes = _lib.load().mts_moe_wide_head_supported
    assert takes(32768, 768, 64, 8) == 1 and takes(1, 4, 17, 1) == 1
    assert not any((takes(32769, 768, 64, 8), takes(64, 768, 16, 2), takes(64, 768, 65, 2), takes(64, 766, 24, 2), takes(64, 768, 24, 9), takes(0, 768, 24, 2)))
