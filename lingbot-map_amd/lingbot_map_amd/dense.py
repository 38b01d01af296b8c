"""Dense (cache-less) attention of whole frames on the paged kernel.

The frame blocks of the aggregator attend within one frame (lingbot_map/layers/block.py:27-101,
lingbot_map/layers/attention.py:446-465: ``F.scaled_dot_product_attention`` over the frame's own
tokens).  The paged kernel covers that case with a trivial row table: every entry names a row
of the caller's own K/V, the pool is never read.
"""
from __future__ import annotations

import ctypes as C
import math
from typing import Dict

import torch
from torch import Tensor

from . import _native as N

_plans: Dict[tuple, tuple] = {}          # (rows, streams, H, D, device) -> (row table, stream descriptors, workspace bytes)
_tails: Dict[tuple, bytes] = {}          # (streams, H, D, dtype) -> what the calls of such a plan have in common
_calls: Dict[tuple, tuple] = {}          # frames_key of a call -> its plan as attend() takes it, and what its addresses belong to
_workspace: Dict[object, Tensor] = {}


def dense_plan(rows: int, num_streams: int, H: int, D: int, device) -> tuple:
    """(row table, stream descriptors, workspace) of ``num_streams`` groups of ``rows / num_streams``
    tokens that attend to themselves; the first two are kept per shape, the workspace per device and
    scratch lane (one chain of launches that may overlap another each)."""
    plan = _plans.get((rows, num_streams, H, D, device))
    if plan is None:
        n = rows // num_streams
        # entry -1 - r names row r of the caller's own K/V
        kv_rows = (-1 - torch.arange(rows, dtype=torch.int32)).to(device)
        streams = (N.AttnStream * num_streams)(*[N.AttnStream(s * n, n, s * n, n) for s in range(num_streams)])
        need = int(N.lib.lbm_attn_workspace_bytes(streams, num_streams, H, D))
        plan = _plans[(rows, num_streams, H, D, device)] = (kv_rows, streams, need)
    kv_rows, streams, need = plan
    lane = (device, N.current_scratch_lane())
    ws = _workspace.get(lane)
    if ws is None or ws.numel() < max(need, 16):
        ws = _workspace[lane] = torch.empty(max(int(need * 1.25), 1 << 20), dtype=torch.uint8, device=device)
    return kv_rows, streams, ws


def _tail(num_streams: int, H: int, D: int, dtype) -> bytes:
    tail = _tails.get((num_streams, H, D, dtype))
    if tail is None:
        tail = _tails[(num_streams, H, D, dtype)] = N.attn_call_tail(
            0, num_streams, H, D, 16, N.DTYPE_BF16 if dtype == torch.bfloat16 else N.DTYPE_F32, N.ATTN_OWN_ROWS)
    return tail


def dense_attention(q: Tensor, k: Tensor, v: Tensor, num_streams: int = 1, q_prescaled: bool = False) -> Tensor:
    """softmax(q k^T / sqrt(D)) v for ``num_streams`` independent token groups.

    ``q``, ``k``, ``v``: ``[num_streams * n, H, D]`` contiguous, bf16 or fp32, on the GPU; group
    ``s`` is rows ``s * n .. (s + 1) * n - 1`` and attends to itself only.  Returns the same
    shape and dtype.  ``q_prescaled``: q already carries 1 / sqrt(D) and log2(e) (a producer run
    with ``q_scale = q_scale_log2(1 / sqrt(D))``).  Raises on anything the HIP kernels do not cover (there is no fallback)."""
    key = N.host.frames_key(q, k, v, num_streams)
    if key is not None:
        call = _calls.get(key)
        if call is None:
            rows, H, D = key[:3]
            kv_rows, streams, _ = dense_plan(rows, num_streams, H, D, q.device)
            call = _calls[key] = (kv_rows.data_ptr(), C.addressof(streams), max(_plans[(rows, num_streams, H, D, q.device)][2], 16), q.device,
                                  1.0 / math.sqrt(D), _tail(num_streams, H, D, q.dtype), (kv_rows, streams))
        rows_at, streams_at, need, device, scale, tail, _ = call
        ws = _workspace.get((device, N.current_scratch_lane()))
        if ws is None or ws.numel() < need:
            ws = dense_plan(key[0], num_streams, key[1], key[2], device)[2]
        out = N.host.attend(q, k, v, k, rows_at, 0, 0, streams_at, ws, 0.0 if q_prescaled else scale, tail)
        if out.__class__ is int:
            N.check(out)
        return out
    # tensors of a subclass, views, or what is refused here
    assert q.is_cuda and q.dim() == 3 and q.shape == k.shape == v.shape, "q, k, v: [tokens, H, D] on the GPU"
    assert q.dtype == k.dtype == v.dtype and q.dtype in (torch.bfloat16, torch.float32), "bf16 or fp32"
    rows, H, D = q.shape
    assert 1 <= num_streams <= N.MAX_STREAMS and rows % num_streams == 0
    q, k, v = q.contiguous(), k.contiguous(), v.contiguous()
    device = q.device
    kv_rows, streams, ws = dense_plan(rows, num_streams, H, D, device)
    tail = _tail(num_streams, H, D, q.dtype)
    out = torch.empty_like(q)
    k_ptr = k.data_ptr()
    N.check(N.lib.lbm_attn_run_call(N.ATTN_CALL_HEAD.pack(
        q.data_ptr(), k_ptr, out.data_ptr(), k_ptr, v.data_ptr(), kv_rows.data_ptr(), 0, 0, C.addressof(streams), ws.data_ptr(),
        ws.numel(), 0.0 if q_prescaled else 1.0 / math.sqrt(D)) + tail, N.stream_handle(device)))
    return out
