"""Routing metadata of few entries, made by one block, against the oracle: bit-exact."""

import numpy as np
import pytest
import torch

from minitrain_amd import _lib
from oracle import moe_oracle as O

pytestmark = pytest.mark.gpu


# around a wave's step and share, the most entries of the block and one token more; experts up to the most of the block and one more
@pytest.mark.parametrize("T,K,E", [(1, 1, 1), (63, 1, 8), (65, 1, 9), (512, 2, 8), (513, 2, 8), (1365, 3, 64), (2047, 2, 16), (2048, 2, 16), (2049, 2, 16), (512, 8, 256),
                                   (512, 8, 257), (1024, 4, 200)])
@pytest.mark.parametrize("spread", ["even", "dropped", "one"])
@pytest.mark.parametrize("permute", [True, False])
def test_few_entries(T, K, E, spread, permute):
    print(f"route one T={T} K={K} E={E} {spread} permute={permute}", flush=True)
    rng = np.random.default_rng(T + E)
    idx = rng.integers(0, E, (T, K)).astype(np.int32)
    if spread == "dropped":
        idx[rng.random((T, K)) < 0.3] = -1
    if spread == "one":
        idx[:] = E - 1
    lib, index, TK = _lib.load(), torch.from_numpy(idx).cuda(), T * K
    i32 = lambda n: torch.full((n + 8,), -9, dtype=torch.int32, device="cuda")
    counts, start, scatter, reverse, gather = i32(E), i32(E + 1), i32(TK), i32(TK), i32(TK)
    size = lib.mts_moe_route_workspace_bytes(T, K, E)
    ws = torch.empty(size, dtype=torch.uint8, device="cuda")
    arrays = [t.data_ptr() if permute else None for t in (scatter, reverse, gather)]
    assert lib.mts_moe_route(index.data_ptr(), T, K, E, 64, counts.data_ptr(), start.data_ptr(), *arrays, None, None, None, ws.data_ptr(), size, _lib.stream_of(index)) == 0
    want = O.routing_metadata(idx, E, 64)
    kept = int(want.expert_start[-1])
    pairs = [(counts, want.counts), (start, want.expert_start)]
    if permute:
        pairs += [(scatter, want.s_scatter_idx[:kept]), (reverse, want.s_reverse_scatter_idx), (gather, want.x_gather_idx[:kept])]
    for got, expected in pairs:
        assert np.array_equal(got[:len(expected)].cpu().numpy(), expected)
        assert (got[len(expected):] == -9).all()
    if not permute:
        assert all((t == -9).all() for t in (scatter, reverse, gather))
