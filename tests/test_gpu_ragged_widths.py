"""Widths that are not whole 64-wide k-tiles on the pipelined kernels: the last k-tile of every GEMM is partly empty."""

import pytest
import torch

from tests.helpers import BF16_TOL, assert_close_scaled, hip_backend, hip_moe_grads, oracle_moe_grads, routed_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,H,E,I,K", [
    (700, 264, 4, 264, 2),      # one 16-byte chunk in the last k-tile of the forward GEMMs and of dO*W2
    (300, 1000, 8, 1368, 2),    # 40 and 24 elements in the last k-tiles, several column tiles
    (257, 320, 3, 680, 1),      # ragged I only
    (129, 712, 5, 128, 3),      # ragged H only, 2I the shortest that is taken
    (64, 1080, 4, 1288, 2),     # a reduction of more than 1024 in dO*W2 (two blocks per CU)
    (4500, 1096, 8, 520, 2),    # dO*W2 on 256 x 256 tiles, every tile cut in two, rows, columns and k-tiles with a remainder
    (12000, 1032, 4, 264, 2),   # the same, whole tiles
    (1, 504, 2, 504, 1)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_ragged_widths(T, H, E, I, K, dtype):
    """The suite's bound for 16-bit results against the fp32-accumulated oracle."""
    print(f"ragged widths T={T} H={H} E={E} I={I} K={K} {dtype}", flush=True)
    case = routed_case(300 + T, T, H, E, I, K, dtype=dtype)
    args = [case[k] for k in ("x", "w1", "w2", "idx", "w", "g")]
    out, grads = hip_moe_grads(*args)
    ref_out, ref_grads = oracle_moe_grads(*args)
    assert_close_scaled(out, ref_out, BF16_TOL, "out")
    for name, a, b in zip(("dx", "dW1", "dW2", "dS"), grads, ref_grads):
        assert_close_scaled(a, b, BF16_TOL, name)


def test_what_lies_behind_a_row_is_not_multiplied():
    """A token with NaN activations poisons its own output only: the chunks behind the end of the reduction, which in
    memory are the next row's, are not read."""
    T, H, E, I = 200, 264, 2, 328
    case = routed_case(5, T, H, E, I, 2)
    ops = hip_backend()
    x = case["x"].cuda()
    args = [case[k].cuda() for k in ("w1", "w2", "idx", "w")]
    clean = ops.fused_moe(x, *args)
    bad = torch.arange(0, T, 3, device="cuda")
    x[bad] = float("nan")
    poisoned = ops.fused_moe(x, *args)
    good = torch.ones(T, dtype=torch.bool, device="cuda")
    good[bad] = False
    assert torch.isnan(poisoned[bad]).all()
    assert torch.equal(poisoned[good], clean[good])
