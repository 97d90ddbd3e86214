"""fp32 activations through the fp32 GEMMs at the edges of their tiles, against the oracle in fp64."""

import pytest
import torch

from minitrain_amd import _lib
from tests.helpers import assert_close_scaled, hip_moe_grads, oracle_moe_grads, routed_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,H,E,I,K", [
    (700, 72, 3, 40, 2),      # many row tiles per expert, the last one partly empty; k-tiles with a remainder
    (257, 64, 4, 130, 2),     # I not a multiple of 4: rows loaded four bytes at a time; column tiles with a remainder
    (129, 36, 70, 24, 2),     # more experts than a wave holds
    (512, 132, 8, 200, 2),    # wider than a column tile, with a remainder of four
    (1500, 520, 3, 1032, 2),  # tiles of 128 x 128 in every GEMM, the last k-tile half empty
    (1300, 513, 2, 1031, 2),  # the same at odd widths
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


def _down(act, w2, starts):
    y = torch.empty(act.shape[0], w2.shape[1], device="cuda")
    es = torch.tensor(starts, dtype=torch.int32, device="cuda")
    _lib.check(_lib.load().mts_moe_fwd_down(act.data_ptr(), w2.data_ptr(), es.data_ptr(), act.shape[0], w2.shape[0], w2.shape[1], act.shape[1], _lib.MTS_F32,
                                            y.data_ptr(), torch.cuda.current_stream().cuda_stream), "down")
    return y.cpu()


def _dw2(d_out, act, starts):
    T, H = d_out.shape
    dw = torch.empty(len(starts) - 1, H, act.shape[1], device="cuda")
    es = torch.tensor(starts, dtype=torch.int32, device="cuda")
    gather = torch.arange(T, dtype=torch.int32, device="cuda")
    _lib.check(_lib.load().mts_moe_bwd_dw2(d_out.data_ptr(), act.data_ptr(), gather.data_ptr(), es.data_ptr(), T, 1, len(starts) - 1, H, act.shape[1], _lib.MTS_F32,
                                           _lib.MTS_F32, dw.data_ptr(), None, 0, torch.cuda.current_stream().cuda_stream), "dw2")
    return dw.cpu()


@pytest.mark.parametrize("R,H,I", [(90, 72, 100), (2700, 1100, 260)])   # both tile sizes
def test_values_that_three_bf16_terms_do_not_hold(R, H, I):
    """Infinities, NaN, the largest and the smallest numbers, denormal ones among them, in single rows and at any place of the
    reduction: what plain products of these values give, and nothing in the other rows.  1e-5 as above; a value is scaled so that its products are
    ordinary numbers."""
    print(f"special fp32 values R={R} H={H} I={I}", flush=True)
    torch.manual_seed(R)
    starts = [0, R // 3, R // 3, R]
    act, w2 = torch.randn(R, I), torch.randn(3, H, I) * 0.05
    act[3, 5], act[R - 1, I - 1], act[40, 0] = float("inf"), float("-inf"), float("nan")
    act[7] *= 2.0 ** -135
    act[8] *= 2.0 ** -70
    act[9, 40] = 3.4e38
    big = w2 * 2.0 ** 90
    big[:, :, 40] = 0.0   # the largest number meets zero there, where its rounding up would give NaN
    got, got_big = _down(act.cuda(), w2.cuda(), starts), _down(act.cuda(), big.cuda(), starts)
    expert = (torch.arange(R) >= starts[2]).long() * 2
    for w, y in ((w2, got), (big, got_big)):
        want = torch.einsum("ri,rhi->rh", act.double(), w.double()[expert]).float()
        for r in range(R):
            a, b = y[r], want[r]
            if r in (3, 40, R - 1):
                assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.isinf(), b.isinf()) and torch.equal(a[a.isinf()], b[b.isinf()]), r
            elif not (r in (7, 8) and w is w2):
                assert_close_scaled(a, b, 1e-5, f"row {r}")
    # weight gradient: a column of d_out is a row of the result
    d_out, act = torch.randn(R, H), torch.randn(R, I)
    d_out[1, 2], d_out[R - 2, 50], act[5, 9] = float("inf"), float("nan"), 2.0 ** -140
    d_out[R // 3:, 4] *= 2.0 ** -90
    act[R // 3:] *= 2.0 ** 80
    dw = _dw2(d_out.cuda(), act.cuda(), starts)
    assert not dw[1].any()
    for e, (lo, hi) in ((0, (0, starts[1])), (2, (starts[2], R))):
        want = (d_out[lo:hi].double().t() @ act[lo:hi].double()).float()
        for h in range(H):
            assert torch.equal(dw[e, h].isnan(), want[h].isnan()), h
            if want[h].isfinite().all():
                assert_close_scaled(dw[e, h], want[h], 1e-5, f"column {h}")


@pytest.mark.parametrize("R", [1, 2, 3, 17])
@pytest.mark.parametrize("M,N", [(72, 100), (1100, 2100)])   # both tile sizes
def test_sums_of_few_terms(R, M, N):
    """A sum of one term is that product rounded once; sums of up to n terms err by no more than a rounding of the running sum for
    each (n * 2^-24 of the terms' sizes), as the fp32 instruction's do."""
    print(f"few fp32 terms R={R} M={M} N={N}", flush=True)
    torch.manual_seed(R + M)

    def check(got, want, size, name):
        if R == 1:
            assert torch.equal(got, want.float()), name
        assert ((got.double() - want).abs() <= R * 2.0 ** -24 * size).all(), name

    d_out, act = torch.randn(R, M), torch.randn(R, N)
    dw = _dw2(d_out.cuda(), act.cuda(), [0, R])[0]
    check(dw, d_out.double().t() @ act.double(), d_out.double().abs().t() @ act.double().abs(), "weight gradient")
    act, w2 = torch.randn(M, R), torch.randn(1, N, R)
    y = _down(act.cuda(), w2.cuda(), [0, M])
    check(y, act.double() @ w2[0].double().t(), act.double().abs() @ w2[0].double().abs().t(), "rows")


@pytest.mark.parametrize("R,H,I", [(90, 72, 100), (2700, 1100, 260)])   # both tile sizes
def test_products_at_the_ends_of_the_range(R, H, I):
    """Products just below the largest number, alone and in a sum, are finite although a value rounded to fewer bits would not be; products
    of two numbers near 2^-60 keep all their bits, the smallest of which lie below the smallest normal number.  1e-5 as above."""
    print(f"ends of the range R={R} H={H} I={I}", flush=True)
    torch.manual_seed(R)
    starts = [0, R]
    below = torch.tensor(1.0 - 2.0 ** -24)
    act, w2 = torch.zeros(R, I), torch.zeros(1, H, I)
    act[0, 7], w2[0, :, 7] = below * 2.0 ** 127, below * 2.0
    act[1, 20:24], w2[0, :, 20:24] = 0.999 * 2.0 ** 64, 0.999 * 2.0 ** 62
    act[2, 40:], w2[0, :, 40:] = torch.randn(I - 40), torch.randn(H, I - 40)
    y = _down(act.cuda(), w2.cuda(), starts)
    want = act.double() @ w2[0].double().t()
    assert want[:3].float().isfinite().all()
    for r in range(4):
        assert_close_scaled(y[r].double(), want[r], 1e-5, f"row {r}")
    near = 2.0 ** -60
    act, w2 = (1 + torch.rand(R, I)) * near, (1 + torch.rand(1, H, I)) * torch.randn(1, H, I).sign() * near
    y = _down(act.cuda(), w2.cuda(), starts)
    assert_close_scaled(y.double() / near / near, (act.double() @ w2[0].double().t()) / near / near, 1e-5, "small products")
    d_out, act = torch.zeros(R, H), torch.zeros(R, I)
    d_out[3:7, 1], act[3:7, 2] = 0.999 * 2.0 ** 64, 0.999 * 2.0 ** 62
    dw = _dw2(d_out.cuda(), act.cuda(), starts)[0]
    assert_close_scaled(dw.double(), d_out.double().t() @ act.double(), 1e-5, "weight gradient")


@pytest.mark.parametrize("T,H,E,I,K,popular", [
    (1, 4, 1, 4, 1, 0.0), (33, 64, 2, 64, 1, 0.0), (257, 64, 4, 132, 2, 3.0), (129, 36, 70, 24, 2, 0.0), (512, 132, 8, 200, 2, 6.0),
    (1500, 520, 3, 1032, 2, 0.0), (2000, 256, 5, 64, 2, 2.0), (40, 260, 64, 516, 3, 0.0)])
def test_gradients_of_one_launch_are_those_of_separate_ones(T, H, E, I, K, popular, monkeypatch):
    """Both tile sizes for either part, experts without rows and with most of them, dX in front of all, some and none of the weight gradients, more experts
    than a wave has lanes, dropped routes: the same sums in the same order."""
    from minitrain_amd.kernels.hip.switches import SWITCHES

    print(f"fp32 gradients in one launch T={T} H={H} E={E} I={I} K={K} popular={popular}", flush=True)
    case = routed_case(50 + T, T, H, E, I, K, dtype=torch.float32, bias=popular * torch.linspace(-1, 1, E))
    idx = case["idx"].clone()
    if T > 1:
        idx[T // 2, 0] = -1
    one = hip_moe_grads(case["x"], case["w1"], case["w2"], idx, case["w"], case["g"])
    monkeypatch.setattr(SWITCHES, "joint_bwd", False)
    several = hip_moe_grads(case["x"], case["w1"], case["w2"], idx, case["w"], case["g"])
    assert torch.equal(one[0], several[0])
    for name, a, b in zip(("dx", "dW1", "dW2", "dS"), one[1], several[1]):
        assert a.isfinite().all() and torch.equal(a, b), name
