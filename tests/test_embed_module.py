"""The decoder's lookup with another module in the place of its embedding table (CPU)."""

import pytest
import torch
from torch import nn

from minitrain_amd.model.decoder import embed


class _Offers:
    def embedding(self, ids, weight, dtype):
        return torch.full((*ids.shape, weight.shape[1]), 7.0, dtype=dtype)


class _Subclass(nn.Embedding):
    pass


@pytest.mark.parametrize("table,own", [
    (nn.Embedding(9, 4), True), (nn.Embedding(9, 4, padding_idx=1), False), (nn.Embedding(9, 4, max_norm=1.0), False), (nn.Embedding(9, 4, sparse=True), False),
    (nn.Embedding(9, 4, scale_grad_by_freq=True), False), (_Subclass(9, 4), False), (nn.Sequential(nn.Embedding(9, 4), nn.Linear(4, 4)), False)])
def test_only_a_plain_table_takes_the_backends_lookup(table, own):
    ids = torch.tensor([[1, 2, 8]])
    with torch.no_grad():
        got = embed(table, ids, torch.bfloat16, _Offers())
        assert got.dtype == torch.bfloat16
        assert torch.equal(got, torch.full((1, 3, 4), 7.0, dtype=torch.bfloat16) if own else table(ids).bfloat16())
