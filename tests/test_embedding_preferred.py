"""Tables and batches whose gradient this framework sums (host code: no GPU)."""

import pytest

from minitrain_amd import _lib


@pytest.mark.parametrize("T,V,H,own", [
    (1, 50257, 768, True), (1, 65536, 4, True), (1 << 18, 8, 4096, True),
    (255, 65537, 768, False), (256, 65537, 768, True), (500, 128256, 4096, False), (501, 128256, 4096, True), (1023, 262144, 768, False), (1024, 262144, 4, True),
    (4096, 393216, 768, False), (65536, 393216, 768, True), (65536, 524288, 512, True), (65535, 524288, 512, False), (65536, 1 << 20, 768, False),
    (1 << 18, 1 << 20, 256, True), (1 << 18, 1 << 20, 252, False),
    (0, 100, 64, False), ((1 << 18) + 1, 100, 64, False), (100, 100, 66, False), (1 << 18, (1 << 20) + 1, 4096, False)])
def test_own_sums_where_they_are_ahead(T, V, H, own):
    assert _lib.load().mts_embedding_bwd_preferred(T, V, H) == own
