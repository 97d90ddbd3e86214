"""Which copies of weights ride in the launches of the layer's head (host code: no GPU)."""

import pytest

from minitrain_amd import _lib

BF16 = _lib.MTS_BF16


@pytest.mark.parametrize("T,H,E,n1,n2,rides", [
    (64, 768, 8, 1 << 20, 1 << 20, False), (65, 768, 8, 1 << 20, 1 << 20, True),   # one block has no second launch
    (4096, 768, 8, 1 << 34, 8, True), (4096, 768, 8, 8, 1 << 34, True),            # more threads than a launch holds ...
    (4096, 768, 8, (1 << 34) + 8, 8, False), (4096, 768, 8, 8, (1 << 34) + 8, False),
    (4096, 768, 64, 1 << 34, 8, True), (4096, 768, 64, (1 << 36) - 8, 8, False)])   # ... of the other head, too
def test_copies_that_fit_a_launch_ride(T, H, E, n1, n2, rides):
    assert _lib.load().mts_moe_head_casts_ride(T, H, E, BF16, n1, n2) == rides
