"""Copies of master weights that ride in the launches of the layer's head, against the plain conversion and the head without them."""

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

_GUARD = 64


class _Cast(ctypes.Structure):
    _fields_ = [("src", ctypes.c_void_p), ("dst", ctypes.c_void_p), ("n", ctypes.c_int64)]


def _head(x, w_r, K, casts):
    from minitrain_amd import _lib

    lib = _lib.load()
    (T, H), E = x.shape, w_r.shape[0]
    name, size = ("mts_moe_head_cast_fwd", lib.mts_moe_head_workspace_bytes(T, K, E)) if E <= 16 else ("mts_moe_wide_head_cast_fwd", lib.mts_moe_wide_head_workspace_bytes(T, E))
    f32, i32 = dict(dtype=torch.float32, device="cuda"), dict(dtype=torch.int32, device="cuda")
    o = [torch.empty(T, E, **f32), torch.empty(T, K, **f32), torch.empty(T, K, **i32), torch.empty(T, K, dtype=x.dtype, device="cuda"), torch.empty(E, **f32),
         torch.empty(1, **f32), torch.empty(1, **f32), torch.empty(E, **i32), torch.empty(1, **f32), torch.empty(E + 7, **f32), torch.empty(E + 1, **i32),
         *(torch.empty(T * K, **i32) for _ in range(3))]
    ws = torch.empty(size, dtype=torch.uint8, device="cuda")
    rc = getattr(lib, name)(x.data_ptr(), w_r.data_ptr(), T, H, E, K, 1, _lib.dtype_code(x.dtype), *[t.data_ptr() for t in o], ws.data_ptr(), size,
                            ctypes.cast(casts, ctypes.c_void_p) if casts is not None else None, _lib.stream_of(x))
    return rc, o


def _weights(n, seed):
    g = torch.Generator().manual_seed(seed)
    w = torch.randn(n, generator=g) * torch.exp2(torch.randint(-30, 30, (n,), generator=g))
    w[:8] = torch.tensor([float("inf"), -float("inf"), float("nan"), 0.0, -0.0, 1e-40, 3.4e38, 65520.0])
    return w.cuda()


# lengths around the values of a block of 256 and of 512 threads; one block of the head (which has no second launch), a few, and all that it has;
# a head that fills the CUs one by one (129 blocks: the copies have their own launch, 257: they ride)
@pytest.mark.parametrize("T,H,E,K,n1,n2,dtype", [
    (1, 64, 8, 2, 8, 8192, torch.bfloat16), (64, 768, 8, 2, 8200, 8, torch.bfloat16), (65, 768, 8, 2, 8184, 8192, torch.bfloat16),
    (65, 760, 16, 1, 8192, 8200, torch.float16), (1000, 64, 8, 2, 40008, 3 * 8192, torch.float16), (20000, 768, 8, 2, 1 << 20, 1 << 19, torch.bfloat16),
    (40000, 64, 4, 2, 8, 8, torch.bfloat16), (2064, 1024, 16, 2, 8200, 8192, torch.float16), (4112, 1024, 16, 2, 8192, 8200, torch.bfloat16), (1, 64, 17, 1, 8, 8, torch.float16), (300, 768, 64, 4, 16384, 16376, torch.bfloat16), (5000, 132, 33, 8, 16392, 8, torch.bfloat16)])
def test_copies_beside_the_head(T, H, E, K, n1, n2, dtype):
    print(f"head with copies T={T} H={H} E={E} K={K} n={n1},{n2} {dtype}", flush=True)
    g = torch.Generator().manual_seed(T)
    x, w_r = torch.randn(T, H, generator=g).to(dtype).cuda(), torch.randn(E, H, generator=g).cuda()
    sources = [_weights(n1, 1), _weights(n2, 2)]
    copies = [torch.full((n + _GUARD,), 7.0, dtype=dtype, device="cuda") for n in (n1, n2)]
    casts = (_Cast * 2)(*(_Cast(s.data_ptr(), d.data_ptr(), s.numel()) for s, d in zip(sources, copies)))
    rc, got = _head(x, w_r, K, casts)
    assert rc == 0
    rc, want = _head(x, w_r, K, None)
    assert rc == 0
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    for source, copy in zip(sources, copies):
        n = source.numel()
        assert (copy[n:] == 7).all()
        plain = source.to(dtype)
        nan = plain.isnan()
        assert torch.equal(copy[:n].isnan(), nan)
        assert torch.equal(copy[:n].view(torch.int16)[~nan], plain.view(torch.int16)[~nan])


def test_copies_that_are_refused():
    x, w_r = torch.randn(70, 64).bfloat16().cuda(), torch.randn(8, 64).cuda()
    w, d = torch.zeros(64, device="cuda"), torch.zeros(64, dtype=torch.bfloat16, device="cuda")
    good = (w.data_ptr(), d.data_ptr(), 64)
    assert _head(x, w_r, 2, (_Cast * 2)(_Cast(*good), _Cast(*good)))[0] == 0
    for bad, code in (((None, good[1], 64), -1), ((good[0], good[1], 60), -2), ((good[0], good[1], 0), -2), ((good[0] + 4, good[1], 32), -5)):
        assert _head(x, w_r, 2, (_Cast * 2)(_Cast(*good), _Cast(*bad)))[0] == code
    assert _head(x.float(), w_r, 2, (_Cast * 2)(_Cast(*good), _Cast(*good)))[0] == -3
