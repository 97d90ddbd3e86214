"""ctypes binding of ``libmts_moe.so`` (declared in ``include/mts_moe.h``).

The library is loaded after torch so that its HIP symbols bind to the runtime
torch already brought into the process.  There is no fallback: a missing library
raises, and so does every non-zero return code.
"""

from __future__ import annotations

import ctypes
import os
import threading

import torch  # noqa: F401  (must be imported before the library is opened)

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "lib", "libmts_moe.so")

MTS_BF16 = 0
MTS_F32 = 1
MTS_F16 = 2

_c = ctypes
_p = _c.c_void_p
_i = _c.c_int
_l = _c.c_int64

# name -> (restype, argtypes); one entry per declaration in include/mts_moe.h
SIGNATURES = {
    "mts_version": (_i, []),
    "mts_error_string": (_c.c_char_p, [_i]),
    "mts_router_workspace_bytes": (_l, [_l, _i]),
    "mts_router_fwd": (_i, [_p, _l, _i, _i, _i, _p, _p, _p, _p, _p, _p, _p, _p, _p, _i, _p, _l, _p]),
    "mts_router_bwd": (_i, [_p, _p, _p, _p, _p, _i, _p, _p, _p, _p, _l, _i, _i, _i, _p, _p]),
    "mts_router_logits_fwd": (_i, [_p, _p, _l, _i, _i, _i, _p, _p]),
    "mts_router_logits_bwd_workspace_bytes": (_l, [_l, _i, _i]),
    "mts_router_logits_bwd": (_i, [_p, _p, _p, _l, _i, _i, _i, _p, _p, _p, _l, _p]),
    "mts_router_wide_supported": (_i, [_i, _i]),
    "mts_router_wide_fwd": (_i, [_p, _p, _l, _i, _i, _i, _p, _p]),
    "mts_router_wide_bwd_workspace_bytes": (_l, [_l, _i, _i]),
    "mts_router_wide_bwd": (_i, [_p, _p, _p, _l, _i, _i, _i, _p, _p, _p, _l, _p]),
    "mts_moe_route_workspace_bytes": (_l, [_l, _i, _i]),
    "mts_moe_router_route_workspace_bytes": (_l, [_l, _i, _i]),
    "mts_moe_router_route": (_i, [_p, _l, _i, _i, _i, _p, _p, _p, _p, _p, _p, _p, _p, _p, _i, _p, _p, _p, _p, _p, _l, _p]),
    "mts_moe_route": (_i, [_p, _l, _i, _i, _i, _p, _p, _p, _p, _p, _p, _p, _p, _p, _l, _p]),
    "mts_moe_route_static": (_i, [_p, _l, _i, _i, _i, _p, _p, _p, _p, _p, _p, _p, _p, _p]),
    "mts_moe_capacity_workspace_bytes": (_l, [_l, _i, _i]),
    "mts_moe_capacity_mask": (_i, [_p, _p, _l, _i, _i, _l, _p, _p, _p, _p, _l, _p]),
    "mts_moe_capacity_compact_workspace_bytes": (_l, [_l, _i]),
    "mts_moe_capacity_compact": (_i, [_p] * 4 + [_l, _i, _i, _l] + [_p] * 6 + [_l, _p]),
    "mts_moe_capacity_weights_fwd": (_i, [_p, _p, _p, _p, _l, _i, _i, _i, _i, _p, _p, _p]),
    "mts_moe_capacity_weights_bwd": (_i, [_p, _p, _p, _l, _i, _i, _i, _p, _p]),
    "mts_moe_stage_weights": (_i, [_p, _i, _p, _i, _i, _l, _l, _i, _p]),
    "mts_moe_cast_weights_pair": (_i, [_p, _p, _l, _p, _p, _l, _i, _p]),
    "mts_moe_fwd_gateup_swiglu": (_i, [_p, _p, _p, _p, _p, _p, _l, _i, _i, _i, _i, _i, _p, _p, _p]),
    "mts_moe_fwd_down": (_i, [_p, _p, _p, _l, _i, _i, _i, _i, _p, _p]),
    "mts_moe_fwd_joint_supported": (_i, [_i, _i, _i]),
    "mts_moe_fwd_joint_preferred": (_i, [_i, _l, _i, _i, _i]),
    "mts_moe_fwd_joint_workspace_bytes": (_l, [_l, _i]),
    "mts_moe_fwd_gateup_down": (_i, [_p] * 7 + [_l, _i, _i, _i, _i, _i, _p, _p, _p, _p, _l, _p]),
    "mts_moe_fwd_few_rows_supported": (_i, [_i, _i, _l, _l, _i, _i, _i]),
    "mts_moe_fwd_few_rows_preferred": (_i, [_i, _i, _l, _l, _i, _i, _i]),
    "mts_moe_fwd_few_rows_preferred_to_ride": (_i, [_i, _l, _l, _i, _i, _i]),
    "mts_moe_fwd_few_rows": (_i, [_p, _p, _p, _i, _p, _p, _p, _p, _l, _i, _i, _i, _i, _i, _p, _p, _p, _p]),
    "mts_moe_few_tokens_supported": (_i, [_i, _i, _l, _i, _i, _i, _i]),
    "mts_moe_few_tokens_preferred": (_i, [_i, _i, _l, _i, _i, _i, _i]),
    "mts_moe_few_tokens_fwd": (_i, [_p, _p, _p, _p, _i, _l, _i, _i, _i, _i, _i, _i] + [_p] * 20),
    "mts_moe_combine": (_i, [_p, _p, _p, _p, _l, _i, _i, _i, _p, _p]),
    "mts_moe_wide_head_supported": (_i, [_l, _i, _i, _i]),
    "mts_moe_wide_head_workspace_bytes": (_l, [_l, _i]),
    "mts_moe_wide_head_fwd": (_i, [_p, _p, _l, _i, _i, _i, _i, _i] + [_p] * 15 + [_l, _p]),
    "mts_moe_wide_head_cast_fwd": (_i, [_p, _p, _l, _i, _i, _i, _i, _i] + [_p] * 15 + [_l, _p, _p]),
    "mts_moe_head_workspace_bytes": (_l, [_l, _i, _i]),
    "mts_moe_head_fwd": (_i, [_p, _p, _l, _i, _i, _i, _i, _i] + [_p] * 14 + [_p, _l, _p]),
    "mts_moe_head_casts_ride": (_i, [_l, _i, _i, _i, _l, _l]),
    "mts_moe_head_cast_fwd": (_i, [_p, _p, _l, _i, _i, _i, _i, _i] + [_p] * 14 + [_p, _l, _p, _p]),
    "mts_moe_head_bwd_workspace_bytes": (_l, [_l, _i, _i]),
    "mts_moe_head_bwd": (_i, [_p] * 11 + [_l, _i, _i, _i, _i, _i, _p, _p, _p, _l, _p]),
    "mts_moe_ds_partials": (_i, [_i]),
    "mts_probe_mfma_sink_bytes": (_l, [_i]),
    "mts_probe_mfma_rate": (_i, [_i, _i, _i, _p, _l, _p, _p]),
    "mts_moe_bwd_weights_as_stored": (_i, [_i, _i, _i]),
    "mts_moe_bwd_dy1": (_i, [_p, _p, _i, _p, _p, _p, _p, _p, _l, _i, _i, _i, _i, _i, _p, _p, _p, _p, _p]),
    "mts_moe_bwd_schedule_bytes": (_l, [_i]),
    "mts_moe_bwd_schedule": (_i, [_p, _l, _i, _p, _p]),
    "mts_moe_bwd_ds": (_i, [_p, _p, _l, _i, _i, _p, _p]),
    "mts_moe_bwd_dx": (_i, [_p, _p, _i, _p, _l, _i, _i, _i, _i, _p, _p]),
    "mts_moe_bwd_dw_workspace_bytes": (_l, [_i, _i, _i, _i]),
    "mts_moe_bwd_dw2": (_i, [_p, _p, _p, _p, _l, _i, _i, _i, _i, _i, _i, _p, _p, _l, _p]),
    "mts_moe_bwd_dw1": (_i, [_p, _p, _p, _p, _l, _i, _i, _i, _i, _i, _i, _p, _p, _l, _p]),
    "mts_moe_bwd_joint_f32_supported": (_i, [_i, _i]),
    "mts_moe_bwd_joint_f32": (_i, [_p] * 9 + [_l, _i, _i, _i, _i] + [_p] * 5),
    "mts_moe_bwd_joint_supported": (_i, [_i, _i, _i]),
    "mts_moe_bwd_joint": (_i, [_p, _p, _p, _p, _p, _p, _p, _p, _p, _l, _i, _i, _i, _i, _i, _i, _p, _p, _p, _p, _p, _l, _p, _l, _p, _p]),
    "mts_moe_bwd_joint_router_supported": (_i, [_i, _l, _i, _i, _i]),
    "mts_moe_bwd_joint_router": (_i, [_p, _p, _p, _p, _p, _p, _p, _p, _p, _l, _i, _i, _i, _i, _i, _i, _p, _p, _p, _p, _p, _l, _p, _l]
                                 + [_p] * 8 + [_i, _p, _p, _p, _p, _l, _p, _p]),
    "mts_rmsnorm_supported": (_i, [_i]),
    "mts_rmsnorm_fwd": (_i, [_p, _p, _p, _l, _i, _c.c_float, _i, _p, _p, _p, _p]),
    "mts_rmsnorm_bwd_workspace_bytes": (_l, [_l, _i]),
    "mts_rmsnorm_bwd": (_i, [_p, _p, _p, _p, _p, _l, _i, _i, _p, _p, _p, _l, _p]),
    "mts_rope": (_i, [_p, _i, _p, _p, _l, _l, _i, _i, _i, _p]),
    "mts_cross_entropy_fwd": (_i, [_p, _p, _l, _i, _l, _i, _p, _p, _p, _p, _p, _p]),
    "mts_cross_entropy_both_supported": (_i, [_i, _i]),
    "mts_cross_entropy_both": (_i, [_p, _p, _l, _i, _l, _i, _p, _p, _p, _p, _p, _p, _l, _p]),
    "mts_cross_entropy_bwd_unless_one": (_i, [_p, _p, _l, _i, _l, _i, _p, _p, _p, _p, _p, _l, _p]),
    "mts_embedding_bwd_supported": (_i, [_l, _l, _l]),
    "mts_embedding_bwd_preferred": (_i, [_l, _l, _l]),
    "mts_embedding_bwd_workspace_bytes": (_l, [_l, _l, _l]),
    "mts_embedding_bwd": (_i, [_p, _p, _l, _i, _i, _i, _p, _p, _l, _p]),
    "mts_linear_rows_supported": (_i, [_i, _l, _i, _i]),
    "mts_linear_fwd_preferred": (_i, [_i, _l, _i, _i]),
    "mts_linear_fwd": (_i, [_p, _p, _l, _i, _i, _i, _p, _p]),
    "mts_linear_dx_preferred": (_i, [_i, _l, _i, _i]),
    "mts_linear_dx": (_i, [_p, _p, _l, _i, _i, _i, _p, _p]),
    "mts_linear_dw_supported": (_i, [_i, _l, _i, _i]),
    "mts_linear_dw_workspace_bytes": (_l, [_l, _i, _i]),
    "mts_linear_dw": (_i, [_p, _p, _l, _i, _i, _i, _p, _p, _l, _p]),
    "mts_linear_rounds_supported": (_i, [_i, _l, _i, _i, _l]),
    "mts_linear_rounds_workspace_bytes": (_l, [_i, _l, _i, _i]),
    "mts_linear_dw_rounds": (_i, [_p, _l, _p, _l, _i, _i, _i, _p, _p, _l, _p]),
    "mts_linear_dx_rounds": (_i, [_p, _l, _p, _l, _i, _i, _i, _p, _p, _l, _p]),
    "mts_attention_supported": (_i, [_l, _i, _l, _i]),
    "mts_attention_fwd": (_i, [_p, _p, _p, _l, _i, _l, _i, _i, _p, _p, _p]),
    "mts_attention_bwd": (_i, [_p, _p, _p, _p, _p, _p, _l, _i, _l, _i, _i, _p, _p, _p, _p, _p]),
    "mts_attention_turned_fwd": (_i, [_p, _p, _p, _p, _p, _l, _i, _l, _i, _i, _p, _p, _p, _p]),
    "mts_attention_turned_bwd": (_i, [_p, _p, _p, _p, _p, _p, _p, _p, _l, _i, _l, _i, _i, _p, _p, _p, _p, _p]),
    "mts_cross_entropy_bwd": (_i, [_p, _p, _l, _i, _l, _i, _p, _p, _p, _p, _p, _p]),
    "mts_layer_means": (_i, [_p, _p, _p, _p, _i, _p, _p]),
    "mts_scalar_sums": (_i, [_p, _i, _p, _p, _p, _p, _i, _p]),
    "mts_grad_norm_workspace_bytes": (_l, [_p, _i]),
    "mts_grad_norm": (_i, [_p, _i, _c.c_float, _p, _p, _p, _l, _p]),
    "mts_adamw_workspace_bytes": (_l, [_i]),
    "mts_adamw": (_i, [_p, _i, _p, _i, _p, _p, _p, _l, _p]),
    "mts_cross_entropy_bwd_pitched": (_i, [_p, _p, _l, _i, _l, _i, _p, _p, _p, _p, _p, _l, _p]),
}


_lib = None
_host = None
_joint_workspace = None
_lock = threading.Lock()


class MtsError(RuntimeError):
    pass


def load():
    """Open the library once and attach the prototypes."""
    global _lib
    if _lib is not None:
        return _lib
    with _lock:
        if _lib is None:
            if not os.path.exists(LIB_PATH):
                raise MtsError(
                    f"{LIB_PATH} is missing: build it with `python -m minitrain_amd.build` "
                    "(there is no fallback for the hip backend)"
                )
            lib = ctypes.CDLL(LIB_PATH)
            for name, (res, args) in SIGNATURES.items():
                fn = getattr(lib, name)
                fn.restype = res
                fn.argtypes = args
            _lib = lib
    return _lib


def host():
    """The native host path (``csrc/host/mts_host.cpp``): contract checks, allocations and autograd nodes."""
    global _host
    if _host is None:
        load()
        try:
            from minitrain_amd.lib import _host as module
        except ImportError as err:
            raise MtsError(f"lib/_host.so does not load ({err}): build it with `python -m minitrain_amd.build` "
                           "(there is no fallback for the hip backend)") from err
        if _joint_workspace is not None:
            module.set_joint_workspace(_joint_workspace)
        _host = module
    return _host


def set_joint_workspace(provider) -> None:
    """``provider(device_index)``: the counters of the joint gate/up + down launch on the current stream of a device."""
    global _joint_workspace
    _joint_workspace = provider
    if _host is not None:
        _host.set_joint_workspace(provider)


def check(code: int, what: str) -> None:
    if code != 0:
        msg = load().mts_error_string(code).decode()
        raise MtsError(f"{what} failed: {msg} (code {code})")


def ptr(t) -> int:
    return 0 if t is None else t.data_ptr()


def stream_of(t) -> int:
    return torch.cuda.current_stream(t.device).cuda_stream


def dtype_code(dt) -> int:
    if dt == torch.bfloat16:
        return MTS_BF16
    if dt == torch.float32:
        return MTS_F32
    if dt == torch.float16:
        return MTS_F16
    raise MtsError(f"unsupported dtype {dt}")
