"""fp32 activations through the fp32 matrix-instruction GEMMs at the edges of their tiles, against the oracle in fp64."""

import pytest
import torch

from tests.helpers import assert_close_scaled, hip_moe_grads, oracle_moe_grads, routed_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,H,E,I,K", [
    (700, 72, 3, 40, 2),      # many row tiles per expert, the last one partly empty; k-tiles with a remainder
    (257, 64, 4, 130, 2),     # I not a multiple of 4: rows loaded four bytes at a time; column tiles with a remainder
    (129, 36, 70, 24, 2),     # more experts than a wave holds
    (512, 132, 8, 200, 2),    # wider than a column tile, with a remainder of four
    (33, 64, 2, 64, 1), (1, 4, 1, 1, 1)])
@pytest.mark.parametrize("wdtype", [torch.float32, torch.bfloat16])
def test_fp32_gemms(T, H, E, I, K, wdtype):
    """1e-5 of a tensor's largest value: fp32 sums of up to a thousand products of either sign (2^-24 * sqrt(1000) = 2e-6);
    gradients of 16-bit weights are rounded once more (2^-9)."""
    print(f"fp32 gemms T={T} H={H} E={E} I={I} K={K} {wdtype}", flush=True)
    case = routed_case(7 + T, T, H, E, I, K, dtype=torch.float32)
    w1, w2 = case["w1"].to(wdtype), case["w2"].to(wdtype)
    out, grads = hip_moe_grads(case["x"], w1, w2, case["idx"], case["w"], case["g"])
    ref_out, ref_grads = oracle_moe_grads(case["x"], w1, w2, case["idx"], case["w"], case["g"], compute_dtype=torch.float64)
    assert_close_scaled(out, ref_out, 1e-5, "out")
    for name, a, b in zip(("dx", "dW1", "dW2", "dS"), grads, ref_grads):
        assert_close_scaled(a, b, 2.0 ** -8 if a.dtype == torch.bfloat16 else 1e-5, name)
