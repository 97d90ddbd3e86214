"""The decoder's operators around its matrix products: RMSNorm, rotary encoding and cross-entropy.

Each stands in for a chain of stock elementwise and reduction kernels
(minitrain/kernels/torch_ops.py of the reference) that reads and writes the activations several
times over, in fp32 on the way: here one launch forward and one or two backward, each operand read
once and each result written once.  The predicates say what the kernels take; the backend leaves
everything else (CPU tensors, other dtypes or layouts) to the stock operators.
"""

import torch

from minitrain_amd import _lib

_ACT = (torch.bfloat16, torch.float16, torch.float32)
_INT_MAX = 2**31 - 1


def _aligned(t):
    """Dense and starting on a 16-byte boundary (a view may start inside an allocation)."""
    t = t.contiguous()
    return t.clone() if t.data_ptr() % 16 else t


# ---- RMSNorm, with the residual sum in front of it -----------------------------------------------

def is_rmsnorm_supported(x, weight, residual=None) -> bool:
    return (
        x.is_cuda and weight.is_cuda and x.dtype in _ACT and weight.dtype == torch.float32 and weight.ndim == 1
        and x.ndim >= 1 and x.shape[-1] == weight.shape[0] and x.numel() > 0
        and (residual is None or (residual.is_cuda and residual.dtype == x.dtype and residual.shape == x.shape and residual.data_ptr() % 16 == 0))
        and x.data_ptr() % 16 == 0 and weight.data_ptr() % 16 == 0   # a view may start inside an allocation
        and bool(_lib.load().mts_rmsnorm_supported(x.shape[-1]))
    )


class _RMSNormFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, residual, weight, eps):
        lib = _lib.load()
        x, weight = x.contiguous(), weight.contiguous()
        H = x.shape[-1]
        N = x.numel() // H
        y = torch.empty_like(x)
        total = x
        if residual is not None:
            residual = residual.contiguous()
            total = torch.empty_like(x)
        rstd = torch.empty(N, dtype=torch.float32, device=x.device)
        _lib.check(
            lib.mts_rmsnorm_fwd(x.data_ptr(), _lib.ptr(residual), weight.data_ptr(), N, H, eps, _lib.dtype_code(x.dtype),
                                total.data_ptr() if residual is not None else None, y.data_ptr(), rstd.data_ptr(), _lib.stream_of(x)),
            "mts_rmsnorm_fwd",
        )
        ctx.save_for_backward(total, weight, rstd)
        ctx.set_materialize_grads(False)
        if residual is None:
            return y
        return total, y

    @staticmethod
    def backward(ctx, *grads):
        g_sum, g_y = grads if len(grads) == 2 else (None, grads[0])
        total, weight, rstd = ctx.saved_tensors
        if g_y is None:   # only the residual stream goes on
            return g_sum, (g_sum if len(grads) == 2 else None), None, None
        lib = _lib.load()
        H = total.shape[-1]
        N = total.numel() // H
        g_y = _aligned(g_y)
        g_sum = None if g_sum is None else _aligned(g_sum)
        d_sum = torch.empty_like(total)
        d_weight = torch.empty_like(weight)
        ws_bytes = lib.mts_rmsnorm_bwd_workspace_bytes(N, H)
        ws = torch.empty(ws_bytes, dtype=torch.uint8, device=total.device)
        _lib.check(
            lib.mts_rmsnorm_bwd(g_y.data_ptr(), _lib.ptr(g_sum), total.data_ptr(), weight.data_ptr(), rstd.data_ptr(), N, H,
                                _lib.dtype_code(total.dtype), d_sum.data_ptr(), d_weight.data_ptr(), ws.data_ptr(), ws_bytes,
                                _lib.stream_of(total)),
            "mts_rmsnorm_bwd",
        )
        return d_sum, (d_sum if len(grads) == 2 else None), d_weight, None


def rmsnorm(x, weight, eps: float):
    return _RMSNormFunction.apply(x, None, weight, eps)


def add_rmsnorm(x, residual, weight, eps: float):
    """``(x + residual, rmsnorm(x + residual))``"""
    return _RMSNormFunction.apply(x, residual, weight, eps)


# ---- rotary encoding -----------------------------------------------------------------------------

_TURN, _TURN_BACK, _COPY = 0, 1, 2


def _launch_rope(jobs, cos, sin, B, S, heads, head_dim, like):
    """``jobs``: (input, output, mode) with both tensors ``[B, heads, S, head_dim]`` of any strides but a dense last dimension."""
    array = (_lib.RopeTensor * len(jobs))()
    for slot, (src, dst, mode) in zip(array, jobs):
        (ib, ih, i_s, _), (ob, oh, os_, _) = src.stride(), dst.stride()
        slot.input, slot.output, slot.mode = src.data_ptr(), dst.data_ptr(), mode
        slot.in_b, slot.in_s, slot.in_h = ib, i_s, ih
        slot.out_b, slot.out_s, slot.out_h = ob, os_, oh
    _lib.check(
        _lib.load().mts_rope(array, len(jobs), cos.data_ptr(), sin.data_ptr(), B, S, heads, head_dim, _lib.dtype_code(like.dtype),
                             _lib.stream_of(like)),
        "mts_rope",
    )


def _table_fits(t, q, S, D):
    return t.is_cuda and t.dtype == q.dtype and tuple(t.shape) == (S, D) and t.is_contiguous() and not t.requires_grad


def is_rope_supported(q, k, cos, sin) -> bool:
    if not (q.is_cuda and k.is_cuda and q.ndim == 4 and q.shape == k.shape and q.dtype == k.dtype and q.dtype in _ACT and q.numel() > 0):
        return False
    B, heads, S, D = q.shape
    return D % 2 == 0 and B * S <= _INT_MAX and _table_fits(cos, q, S, D) and _table_fits(sin, q, S, D)


def _dense_rows(t):
    return t if t.stride(-1) == 1 else t.contiguous()


class _RopeFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, cos, sin):
        q, k = _dense_rows(q), _dense_rows(k)
        B, heads, S, D = q.shape
        # [B, S, heads, D] in memory, as the projection that q and k are views of
        out = [torch.empty(B, S, heads, D, dtype=q.dtype, device=q.device).transpose(1, 2) for _ in range(2)]
        _launch_rope([(q, out[0], _TURN), (k, out[1], _TURN)], cos, sin, B, S, heads, D, q)
        ctx.save_for_backward(cos, sin)
        return out[0], out[1]

    @staticmethod
    def backward(ctx, g_q, g_k):
        cos, sin = ctx.saved_tensors
        g_q, g_k = _dense_rows(g_q), _dense_rows(g_k)
        B, heads, S, D = g_q.shape
        out = [torch.empty(B, S, heads, D, dtype=g_q.dtype, device=g_q.device).transpose(1, 2) for _ in range(2)]
        _launch_rope([(g_q, out[0], _TURN_BACK), (g_k, out[1], _TURN_BACK)], cos, sin, B, S, heads, D, g_q)
        return out[0], out[1], None, None


def rope(q, k, cos, sin):
    return _RopeFunction.apply(q, k, cos, sin)


class _QkvRopeFunction(torch.autograd.Function):
    """Packed projection ``[B, S, 3 * heads * D]`` to rotated queries, rotated keys and values ``[B, heads, S, D]``.  The
    values stay where they are; the backward launch writes the gradient of the projection in one piece."""

    @staticmethod
    def forward(ctx, qkv, cos, sin, heads):
        qkv = qkv.contiguous()
        B, S, width = qkv.shape
        D = width // (3 * heads)
        q, k, v = (t.transpose(1, 2) for t in qkv.view(B, S, 3, heads, D).unbind(2))
        out = [torch.empty(B, S, heads, D, dtype=qkv.dtype, device=qkv.device).transpose(1, 2) for _ in range(2)]
        _launch_rope([(q, out[0], _TURN), (k, out[1], _TURN)], cos, sin, B, S, heads, D, qkv)
        ctx.save_for_backward(cos, sin)
        ctx.dims = (B, S, heads, D)
        ctx.set_materialize_grads(False)
        return out[0], out[1], v

    @staticmethod
    def backward(ctx, g_q, g_k, g_v):
        cos, sin = ctx.saved_tensors
        B, S, heads, D = ctx.dims
        given = [g for g in (g_q, g_k, g_v) if g is not None]
        if not given:
            return None, None, None, None
        # a zero gradient for a part that took no part in the loss
        fill = torch.empty if len(given) == 3 else torch.zeros
        g_qkv = fill(B, S, 3, heads, D, dtype=given[0].dtype, device=given[0].device)
        jobs = []
        for i, (g, mode) in enumerate(((g_q, _TURN_BACK), (g_k, _TURN_BACK), (g_v, _COPY))):
            if g is not None:
                jobs.append((_dense_rows(g), g_qkv[:, :, i].transpose(1, 2), mode))
        _launch_rope(jobs, cos, sin, B, S, heads, D, given[0])
        return g_qkv.view(B, S, 3 * heads * D), None, None, None


def is_qkv_rope_supported(qkv, cos, sin, heads: int) -> bool:
    if not (qkv.is_cuda and qkv.ndim == 3 and qkv.dtype in _ACT and qkv.numel() > 0 and qkv.shape[-1] % (3 * heads) == 0):
        return False
    B, S, width = qkv.shape
    D = width // (3 * heads)
    return D % 2 == 0 and B * S <= _INT_MAX and _table_fits(cos, qkv, S, D) and _table_fits(sin, qkv, S, D)


def qkv_rope(qkv, cos, sin, heads: int):
    return _QkvRopeFunction.apply(qkv, cos, sin, heads)


# ---- cross-entropy -------------------------------------------------------------------------------

_IGNORE_INDEX = -100   # torch's default


def is_cross_entropy_supported(logits, targets) -> bool:
    return (
        logits.is_cuda and targets.is_cuda and logits.ndim == 2 and targets.ndim == 1 and logits.dtype in _ACT
        and targets.dtype == torch.int64 and logits.shape[0] == targets.shape[0] and 0 < logits.shape[0] <= _INT_MAX
        and 0 < logits.shape[1] <= _INT_MAX
    )


class _CrossEntropyFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, logits, targets):
        logits, targets = _aligned(logits), targets.contiguous()
        N, V = logits.shape
        rows = torch.empty(3, N, dtype=torch.float32, device=logits.device)
        scalars = torch.empty(2, dtype=torch.float32, device=logits.device)
        row_max, row_log_sum, row_loss = rows.unbind(0)
        loss, inv_count = scalars[0], scalars[1]
        _lib.check(
            _lib.load().mts_cross_entropy_fwd(logits.data_ptr(), targets.data_ptr(), N, V, _IGNORE_INDEX, _lib.dtype_code(logits.dtype),
                                              row_max.data_ptr(), row_log_sum.data_ptr(), row_loss.data_ptr(), loss.data_ptr(), inv_count.data_ptr(),
                                              _lib.stream_of(logits)),
            "mts_cross_entropy_fwd",
        )
        ctx.save_for_backward(logits, targets, row_max, row_log_sum, inv_count)
        return loss

    @staticmethod
    def backward(ctx, g_loss):
        logits, targets, row_max, row_log_sum, inv_count = ctx.saved_tensors
        N, V = logits.shape
        g_loss = g_loss.to(torch.float32).contiguous()
        d_logits = torch.empty_like(logits)
        _lib.check(
            _lib.load().mts_cross_entropy_bwd(logits.data_ptr(), targets.data_ptr(), N, V, _IGNORE_INDEX, _lib.dtype_code(logits.dtype),
                                              row_max.data_ptr(), row_log_sum.data_ptr(), g_loss.data_ptr(), inv_count.data_ptr(), d_logits.data_ptr(),
                                              _lib.stream_of(logits)),
            "mts_cross_entropy_bwd",
        )
        return d_logits, None


def cross_entropy(logits, targets):
    """``F.cross_entropy(logits.float(), targets)`` without the fp32 copy of the logits"""
    return _CrossEntropyFunction.apply(logits, targets)
