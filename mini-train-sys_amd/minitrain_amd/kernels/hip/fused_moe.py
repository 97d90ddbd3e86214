"""Fused top-k MoE (dispatch -> grouped SwiGLU experts -> weighted combine).

Counterpart of minitrain/kernels/triton/fused_moe.py:37-449: the support predicate, the
routing-metadata step and the module-level entry point.  The contract checks, the allocations and
the autograd node are native (``csrc/host/mts_host.cpp``); nothing synchronises with the host.
"""

import warnings

import torch

from minitrain_amd import _lib
from minitrain_amd.kernels.hip.switches import SWITCHES

BLOCK_M_TOKEN = 64


def _all_tensors(*args) -> bool:
    return all(isinstance(a, torch.Tensor) for a in args)


def fused_moe_violation(x, gate_up_proj, down_proj, top_k_index, top_k_weights):
    """The first requirement of the operator's tensor contract that the arguments miss, or None."""
    if not _all_tensors(x, gate_up_proj, down_proj):
        return "x, gate_up_proj and down_proj are tensors"
    if not _all_tensors(top_k_index, top_k_weights):
        return "top_k_index and top_k_weights are tensors"
    return _lib.host().fused_moe_violation(x, gate_up_proj, down_proj, top_k_index, top_k_weights)


def is_fused_moe_supported(x, gate_up_proj, down_proj, top_k_index, top_k_weights) -> bool:
    """Counterpart of the reference's predicate (minitrain/kernels/triton/fused_moe.py:37-71)."""
    return fused_moe_violation(x, gate_up_proj, down_proj, top_k_index, top_k_weights) is None


def compute_routing_metadata(topk_indices: torch.Tensor, E: int, block_m_token: int = BLOCK_M_TOKEN):
    """Counts, expert offsets, the stable expert-major permutation and the tile list.

    Returns the same eight tensors, in the same order, as the reference's
    ``compute_routing_metadata`` (minitrain/kernels/triton/fused_moe.py:74-154).
    """
    lib = _lib.load()
    topk_indices = topk_indices.contiguous()
    T, K = topk_indices.shape
    TK = T * K
    dev = topk_indices.device
    i32 = dict(dtype=torch.int32, device=dev)
    expert_token_count = torch.empty(E, **i32)
    expert_start_idx = torch.empty(E + 1, **i32)
    s_scatter_idx = torch.empty(TK, **i32)
    s_reverse_scatter_idx = torch.empty(TK, **i32)
    x_gather_idx = torch.empty(TK, **i32)
    max_m_tiles = min(TK, -(-TK // block_m_token) + E - 1)
    tile_row_start = torch.empty(max_m_tiles, **i32)
    tile_expert = torch.empty(max_m_tiles, **i32)
    tile_count = torch.empty(1, **i32)
    ws_bytes = lib.mts_moe_route_workspace_bytes(T, K, E)
    ws = torch.empty(max(ws_bytes, 4), dtype=torch.uint8, device=dev)
    _lib.check(
        lib.mts_moe_route(
            topk_indices.data_ptr(), T, K, E, block_m_token, expert_token_count.data_ptr(),
            expert_start_idx.data_ptr(), s_scatter_idx.data_ptr(), s_reverse_scatter_idx.data_ptr(),
            x_gather_idx.data_ptr(), tile_row_start.data_ptr(), tile_expert.data_ptr(),
            tile_count.data_ptr(), ws.data_ptr(), ws_bytes, _lib.stream_of(topk_indices),
        ),
        "mts_moe_route",
    )
    return (
        expert_token_count,
        expert_start_idx,
        x_gather_idx,
        s_scatter_idx,
        s_reverse_scatter_idx,
        tile_row_start,
        tile_expert,
        tile_count,
    )


def routing_for_experts(topk_indices: torch.Tensor, E: int):
    """``(expert_start, x_gather, s_scatter, s_reverse)``: what the operator itself needs of the routing
    metadata (the tile list of the reference's kernels is not produced)."""
    return _lib.host().route(topk_indices, E)


def expert_counts(topk_indices: torch.Tensor, E: int) -> torch.Tensor:
    """Routes per expert, int32 ``[E]``: the histogram pass of the routing metadata alone.

    Stands in for ``torch.bincount(expert_indices.flatten().long(), minlength=E)`` of the
    router module (minitrain/model/moe_router.py:82) without its host synchronisation.
    """
    lib = _lib.load()
    topk_indices = topk_indices.contiguous()
    if topk_indices.dtype != torch.int32 or topk_indices.ndim != 2 or not topk_indices.is_cuda:
        raise RuntimeError("hip expert_counts requires a 2D int32 index tensor on the GPU")
    T, K = topk_indices.shape
    dev = topk_indices.device
    out = torch.empty(2 * E + 1, dtype=torch.int32, device=dev)   # counts, then expert_start
    ws_bytes = lib.mts_moe_route_workspace_bytes(T, K, E)
    ws = torch.empty(max(ws_bytes, 4), dtype=torch.uint8, device=dev)
    _lib.check(
        lib.mts_moe_route(
            topk_indices.data_ptr(), T, K, E, BLOCK_M_TOKEN, out.data_ptr(), out[E:].data_ptr(), None, None, None,
            None, None, None, ws.data_ptr(), ws_bytes, _lib.stream_of(topk_indices),
        ),
        "mts_moe_route",
    )
    return out[:E]


# The weight-gradient GEMMs cut the rows of an over-full expert into chunks when they are given a
# workspace for the chunk partials (skewed routing); beyond this size they run without one.
_DW_WORKSPACE_LIMIT = 512 * 2**20


_seen_shapes: set = set()


def dw_workspace_limit(x, gate_up_proj) -> int:
    """The limit to hand to the native side; says once per shape when it leaves the backward pass without row chunks."""
    E, two_i, H = gate_up_proj.shape
    if (E, H, two_i) not in _seen_shapes and x.dtype != torch.float32 and torch.is_grad_enabled():
        # from here on an over-full expert is not cut into row chunks and the joint launch gets no schedule, so skewed routing
        # costs these widths more time than it has to (the results are the same)
        _seen_shapes.add((E, H, two_i))
        nbytes = max(_lib.load().mts_moe_bwd_dw_workspace_bytes(which, E, H, two_i // 2) for which in (1, 2))
        if nbytes > _DW_WORKSPACE_LIMIT:
            warnings.warn(f"hip fused MoE: the row-chunk workspace of the weight-gradient GEMMs for E={E}, H={H}, I={two_i // 2} would take "
                          f"{nbytes / 2**20:.0f} MiB (limit {_DW_WORKSPACE_LIMIT / 2**20:.0f} MiB); running without it", RuntimeWarning,
                          stacklevel=3)
    return _DW_WORKSPACE_LIMIT


class _JointForwardWorkspace:
    """Counters of the launch that holds gate/up and down (``mts_moe_fwd_gateup_down``), one per device and stream.

    The launch needs them zero and leaves them zero, so the layers of a model that run one after the other on a stream
    share one buffer.  Word 0 is the launch's status: it stays zero unless a block gave up waiting for the rows it reads
    (or found them written on another XCD than its own); the outputs of that call are then invalid.  Nothing here
    waits for the GPU: every ``CHECK_EVERY`` calls the word is copied to pinned host memory, and the copy of an earlier
    call is looked at once its event has passed, so an error is raised a few calls late rather than never."""

    CHECK_EVERY = 16

    def __init__(self, device: torch.device):
        self.device = device
        self.buf = None
        self.host = None     # pinned word, allocated with the first copy (not while a graph is being captured)
        self.event = None
        self.calls = 0

    def get(self, nbytes: int) -> torch.Tensor:
        if self.buf is None or self.buf.numel() * 4 < nbytes:
            self.buf = torch.zeros((nbytes + 3) // 4, dtype=torch.int32, device=self.device)
        return self.buf

    def _raise(self, status: int):
        self.buf = None     # the counters of a failed launch are not trusted again
        raise RuntimeError(f"hip fused MoE: the joint gate/up + down launch reported status {status} "
                           "(1: a block gave up waiting for its rows, 2: rows written on another XCD); the outputs of "
                           "that call are invalid. MTS_NO_JOINT_FWD=1 runs the two GEMMs as launches of their own.")

    def before_launch(self):
        # (a stream that is being captured into a graph admits neither the query nor the copy: the word is then left
        # to joint_forward_status())
        if torch.cuda.is_current_stream_capturing():
            return
        if self.event is not None and self.event.query():
            self.event = None
            if int(self.host[0]) != 0:
                self._raise(int(self.host[0]))

    def after_launch(self):
        self.calls += 1
        if torch.cuda.is_current_stream_capturing():
            return
        if self.event is None and self.calls % self.CHECK_EVERY == 1:
            if self.host is None:
                self.host = torch.zeros(1, dtype=torch.int32, pin_memory=True)
            self.host.copy_(self.buf[:1], non_blocking=True)
            self.event = torch.cuda.Event()
            self.event.record()

    def status(self) -> int:
        """The status word now (waits for the stream)."""
        return 0 if self.buf is None else int(self.buf[0].item())


_JOINT_FWD: dict = {}


def _joint_forward_workspace(device: torch.device) -> _JointForwardWorkspace:
    key = (device.index if device.index is not None else torch.cuda.current_device(), torch.cuda.current_stream(device).cuda_stream)
    ws = _JOINT_FWD.get(key)
    if ws is None:
        ws = _JOINT_FWD[key] = _JointForwardWorkspace(device)
    return ws


_lib.set_joint_workspace(lambda index: _joint_forward_workspace(torch.device("cuda", index)))


def joint_forward_status(device=None) -> int:
    """Status of the joint gate/up + down launches on the current stream of ``device`` (0: all of them ran through).
    Synchronises; for tests, benchmarks and the points where a training loop reads a value back anyway."""
    device = torch.device("cuda", torch.cuda.current_device()) if device is None else torch.device(device)
    return _joint_forward_workspace(device).status()


def _width_granule(dtype: torch.dtype) -> int:
    """The kernels move 16 bytes per lane: rows must be a whole number of 16-byte chunks."""
    return 4 if dtype == torch.float32 else 8


def _padded_operands(x, gate_up_proj, down_proj):
    """Zero-padded copies whose widths are whole 16-byte chunks: H -> H8 everywhere, I -> I8 with the gate
    rows at 0.. and the up rows at I8...  Zero columns and rows contribute nothing to any product, so the
    operator's result on the padded operands, cut back to H columns, is the result on the originals; the
    copies are made with differentiable torch ops, so the gradients come back cut to size as well."""
    g = _width_granule(x.dtype)
    E, two_i, H = gate_up_proj.shape
    I = two_i // 2
    H8 = -(-H // g) * g
    I8 = I if x.dtype == torch.float32 else -(-I // g) * g
    pad = torch.nn.functional.pad
    gate, up = gate_up_proj[:, :I], gate_up_proj[:, I:]
    w1 = torch.cat([pad(gate, (0, H8 - H, 0, I8 - I)), pad(up, (0, H8 - H, 0, I8 - I))], dim=1)
    return pad(x, (0, H8 - H)), w1, pad(down_proj, (0, I8 - I, 0, H8 - H))


def fused_moe(x, gate_up_proj, down_proj, top_k_index, top_k_weights):
    missed = fused_moe_violation(x, gate_up_proj, down_proj, top_k_index, top_k_weights)
    if missed is not None:
        raise RuntimeError(f"Unsupported tensor contract for hip fused MoE: it requires {missed}")
    host = _lib.host()
    if host.needs_padding(x, gate_up_proj):
        # widths that are not whole 16-byte chunks (legal in the reference, minitrain/kernels/triton/fused_moe.py:55-70)
        H = x.shape[1]
        xp, w1p, w2p = _padded_operands(x, gate_up_proj, down_proj)
        return host.fused_moe(xp, w1p, w2p, top_k_index, top_k_weights, SWITCHES.mask(), dw_workspace_limit(xp, w1p))[:, :H]
    return host.fused_moe(x, gate_up_proj, down_proj, top_k_index, top_k_weights, SWITCHES.mask(), dw_workspace_limit(x, gate_up_proj))
