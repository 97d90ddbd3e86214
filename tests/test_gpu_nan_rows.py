"""Rows whose router logits are all NaN: their routes have rows of their own, and no other token notices them."""

import pytest
import torch

from oracle import moe_oracle as O
from tests.helpers import hip_backend
from tests.test_gpu_head_casts import _head

pytestmark = pytest.mark.gpu


def _with_bad_rows(T, H, E, dtype, fill):
    """Every fifth token is bad, and behind each comes one that prefers the last expert."""
    x, w_r, _, _, _ = O.make_inputs(T + E, T, H, E, 8)
    bad = torch.arange(T) % 5 == 1
    x[2::5] = 4 * w_r[E - 1] / w_r[E - 1].norm()
    x[bad] = fill
    return x.to(dtype).cuda(), w_r.cuda(), bad


# one block of the head, a few, the heads of few experts on either pipe, the chained head of many
@pytest.mark.parametrize("T,H,E,K,dtype", [
    (40, 64, 8, 2, torch.bfloat16), (600, 64, 8, 2, torch.bfloat16), (600, 60, 7, 3, torch.bfloat16), (600, 64, 16, 8, torch.float16),
    (2, 64, 17, 1, torch.float16), (600, 64, 24, 4, torch.bfloat16), (333, 132, 64, 8, torch.bfloat16)])
def test_counters_and_scatter_agree(T, H, E, K, dtype):
    print(f"bad rows T={T} H={H} E={E} K={K} {dtype}", flush=True)
    from minitrain_amd.kernels.hip.fused_moe import compute_routing_metadata
    from minitrain_amd.kernels.hip.router import router_logits, router_postprocess

    x, w_r, bad = _with_bad_rows(T, H, E, dtype, float("nan"))
    rc, got = _head(x, w_r, K, None)
    assert rc == 0
    indices, counts, start, scatter, reverse, gather = got[2], got[7], *got[10:]
    route = router_postprocess(router_logits(x, w_r), K, normalize=True)
    assert torch.equal(indices, route.expert_indices) and torch.equal(counts, route.expert_counts)
    assert torch.equal(indices[bad.cuda()].cpu(), torch.arange(K, dtype=torch.int32).expand(int(bad.sum()), K))
    want = compute_routing_metadata(indices, E)
    for name, a, b in zip(("counts", "expert_start", "x_gather", "s_scatter", "s_reverse"), (counts, start, gather, scatter, reverse), want):
        assert torch.equal(a, b), name


@pytest.mark.parametrize("E,K", [(4, 2), (24, 3), (80, 2)])
@pytest.mark.parametrize("limited", [False, True])
def test_other_tokens_do_not_notice(E, K, limited):
    """Against tokens of zeros in the place of the bad ones, whose routes are the same: the first K of experts that tie."""
    from minitrain_amd.model.blocks import MoEFeedForward
    from minitrain_amd.model.config import ModelConfig

    print(f"bad rows in a layer E={E} K={K} limited={limited}", flush=True)
    T, H, I = 600, 64, 64
    torch.manual_seed(E)
    block = MoEFeedForward(ModelConfig(n_layers=1, n_heads=1, hidden_size=H, intermediate_size=I, num_experts=E, experts_per_token=K,
                                       expert_capacity_factor=float(E) if limited else None)).cuda().eval()   # nothing is dropped
    results = []
    for fill in (float("nan"), 0.0):
        x, w_r, bad = _with_bad_rows(T, H, E, torch.bfloat16, fill)
        with torch.no_grad():
            block.router.weight.copy_(w_r)
            results.append(block(x, hip_backend()).hidden_states)
    bad = bad.cuda()
    assert results[0][bad].isnan().all() and torch.equal(results[0][~bad], results[1][~bad])
