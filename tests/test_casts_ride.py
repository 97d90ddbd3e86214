"""Which copies of weights ride in the launches of the layer's head (host code: no GPU)."""

import pytest

from minitrain_amd import _lib

BF16, FP16 = _lib.MTS_BF16, _lib.MTS_F16


@pytest.mark.parametrize("T,H,E,n1,n2,rides", [
    (64, 768, 8, 1 << 20, 1 << 20, False), (65, 768, 8, 1 << 20, 1 << 20, True),   # one block has no second launch
    (4096, 768, 8, 1 << 34, 8, True), (4096, 768, 8, 8, 1 << 34, True),            # more threads than a launch holds ...
    (4096, 768, 8, (1 << 34) + 8, 8, False), (4096, 768, 8, 8, (1 << 34) + 8, False),
    (4096, 768, 64, 1 << 34, 8, True), (4096, 768, 64, (1 << 36) - 8, 8, False)])   # ... of the other head, too
def test_copies_that_fit_a_launch_ride(T, H, E, n1, n2, rides):
    assert _lib.load().mts_moe_head_casts_ride(T, H, E, BF16, n1, n2) == rides


@pytest.mark.parametrize("T,H,E,dtype,rides", [
    (98304, 1024, 8, BF16, True), (98304, 1024, 12, FP16, True),              # room for two blocks a CU, however many there are
    (8192, 2048, 8, BF16, True), (8193, 2048, 8, BF16, False),                # room for one: 128 blocks of 64 rows leave half of the CUs, 129 do not
    (2048, 1024, 16, BF16, True), (2064, 1024, 16, FP16, False), (4096, 1024, 16, BF16, False), (4112, 1024, 16, BF16, True),   # 16 rows a block
    (6144, 1024, 16, BF16, True), (6160, 1024, 16, BF16, False), (98304, 4096, 8, BF16, False),   # the second round, and all blocks that there are
    (32768, 8192, 64, BF16, True)])
def test_copies_ride_where_the_head_leaves_places(T, H, E, dtype, rides):
    assert _lib.load().mts_moe_head_casts_ride(T, H, E, dtype, 1 << 20, 1 << 20) == rides
