"""ctypes binding of the C ABI declared in include/lbm_paged_attn.h.

There is no CPU fallback: importing this module without the built library raises."""
from __future__ import annotations

import contextlib
import ctypes as C
import importlib.machinery
import importlib.util
import os
import struct

from .build import HOST_PATH, LIB_PATH

OK, ERR_INVALID, ERR_UNSUPPORTED, ERR_WORKSPACE, ERR_HIP = 0, 1, 2, 3, 4
DTYPE_BF16, DTYPE_F32 = 0, 1
LAYOUT_TWO_STREAM, LAYOUT_FRAME_PAGES = 0, 1
ROPE_INTERLEAVED, ROPE_HALF_SPLIT = 0, 1
LINEAR_BIAS, LINEAR_BIAS_GELU, LINEAR_BIAS_RESIDUAL = 0, 1, 2
MAX_STREAMS = 16
MAX_GROUPS = 32
STATIC_SCRATCH_MIB = 64
OP_RESET, OP_ROLLBACK, OP_APPEND, OP_EVICT, OP_PLAN, OP_PLAN_NEWEST_SELF = 1, 2, 4, 8, 16, 32
TERR_NAMES = {1: "patch page pool exhausted", 2: "special page pool exhausted", 4: "window ring full",
              8: "trajectory memory full", 16: "rollback underflow", 32: "visible token count mismatch"}
HDR = {"frame_count": 0, "n_anchor": 1, "win_head": 2, "win_count": 3, "n_free_patch": 4,
       "n_free_special": 5, "n_special_pages": 6, "special_tokens": 7, "n_memory": 8,
       "n_memory_pages": 9, "error": 10, "plan_kv_tokens": 11, "plan_n_pages": 12}
HDR_WORDS = 16
ABI_VERSION = 13


# Scratch memory that the package keeps per device (the K-split workspace of the GEMM, the
# workspace of the cache-less attention) serves one chain of launches at a time.  Code that runs a
# second chain which may overlap the first on the same GPU (another branch of a HIP graph) runs it
# under ``scratch_lane(1)``: every lane has scratch areas of its own.
_scratch_lane = 0


def current_scratch_lane() -> int:
    return _scratch_lane


@contextlib.contextmanager
def scratch_lane(lane: int):
    global _scratch_lane
    before, _scratch_lane = _scratch_lane, int(lane)
    try:
        yield
    finally:
        _scratch_lane = before


class CacheGeom(C.Structure):
    _fields_ = [(n, C.c_int32) for n in (
        "layout", "tokens_per_frame", "num_special_tokens", "page_size", "scale_frames",
        "patch_pages", "special_pages", "memory_frames", "pages_per_stream")]


class StepOp(C.Structure):
    _fields_ = [(n, C.c_int32) for n in (
        "ops", "sliding_window", "keep_tokens", "self_tokens", "q_begin", "kv_row_begin",
        "expect_kv_tokens", "page_out_begin")]


class AttnStream(C.Structure):
    _fields_ = [(n, C.c_int32) for n in ("q_begin", "q_rows", "kv_row_begin", "kv_tokens", "live_at")]


# ``lbm_attn_call`` as two packed pieces, which the caller puts one behind the other: what differs from call to
# call (nine addresses, 0 for none, the workspace's address and size, the softmax scale) and what a plan's calls
# have in common (``attn_call_tail``).  0.5 us a call; eighteen arguments one by one take the binding 2.7.
ATTN_CALL_HEAD = struct.Struct("10PNf")
ATTN_OWN_ROWS, ATTN_APPEND_APART, ATTN_FIXED_ORDER = 1, 2, 4


def attn_call_tail(append_tokens: int, n_streams: int, num_heads: int, head_dim: int, page_size: int, dtype: int, flags: int) -> bytes:
    return struct.pack("7i", append_tokens, n_streams, num_heads, head_dim, page_size, dtype, flags)


class RowNorm(C.Structure):
    """``lbm_row_norm``: a LayerNorm folded into the launch that consumes its output."""
    _fields_ = [("stats", C.c_void_p), ("w_colsum", C.c_void_p), ("stats_tiles", C.c_int32), ("eps", C.c_float)]


class BlockWeights(C.Structure):
    """``lbm_block_weights``: a transformer block's parameters, pointers to device memory."""
    _fields_ = [(n, C.c_void_p) for n in (
        "qkv_w", "proj_w", "fc1_w", "fc2_w", "qkv_b", "proj_b", "fc1_b", "fc2_b", "qkv_colsum", "fc1_colsum", "ls1", "ls2",
        "q_norm_w", "q_norm_b", "k_norm_w", "k_norm_b")] + [(n, C.c_float) for n in ("norm1_eps", "norm2_eps", "qk_eps")] + \
        [(n, C.c_int32) for n in ("num_heads", "hidden")]


class BlockCall(C.Structure):
    """``lbm_block_call``: one pass of a block."""
    _fields_ = [(n, C.c_void_p) for n in (
        "x", "a", "stats", "out", "out_stats", "scratch", "rope_cs", "pool", "append_rows", "kv_rows", "live_kv_tokens",
        "streams", "attn_workspace", "split_workspace")] + \
        [(n, C.c_size_t) for n in ("scratch_bytes", "attn_workspace_bytes", "split_workspace_bytes")] + [("q_scale", C.c_float)] + \
        [(n, C.c_int32) for n in ("rows", "stats_tiles", "rope_layout", "keep_kv", "n_streams", "page_size")] + \
        [("hints", C.c_void_p * 4), ("hint_bytes", C.c_size_t * 4), ("own_rows", C.c_int32)]


SYMBOLS = ("lbm_abi_version", "lbm_last_error", "lbm_tables_words", "lbm_tables_step",
           "lbm_rows_from_pages", "lbm_kv_append", "lbm_qkv_prepare", "lbm_residual_norm", "lbm_linear", "lbm_linear_norm", "lbm_linear_stats_tiles", "lbm_linear_workspace_bytes", "lbm_linear_prefetch_hint", "lbm_qkv_linear_prepare", "lbm_qkv_linear_prepare_norm", "lbm_attn_workspace_bytes", "lbm_attn_run", "lbm_attn_run_append", "lbm_attn_run_live", "lbm_attn_run_call",
           "lbm_attn_run_static", "lbm_block_scratch_bytes", "lbm_block_run",
           "lbm_group_outputs", "lbm_stream_table", "lbm_normalise_images", "lbm_patch_tokens")


def _load():
    if not os.path.exists(LIB_PATH):
        raise RuntimeError(
            f"HIP library {LIB_PATH} is not built; run `python -c 'import __graft_entry__ as g; g.build()'` "
            "(there is no CPU fallback for this path)")
    # torch's libraries first, its HIP runtime among them: loaded before it, the library brings ROCm's own, and of two
    # runtimes in a process one finds no device
    import torch  # noqa: F401
    lib = C.CDLL(LIB_PATH)
    p, i32, vp = C.POINTER, C.c_int32, C.c_void_p
    lib.lbm_abi_version.restype = C.c_int
    lib.lbm_last_error.restype = C.c_char_p
    lib.lbm_tables_words.restype = C.c_int64
    lib.lbm_tables_words.argtypes = [p(CacheGeom)]
    lib.lbm_tables_step.restype = C.c_int
    lib.lbm_tables_step.argtypes = [vp, p(CacheGeom), i32, p(StepOp), vp, vp, vp, vp, vp]
    lib.lbm_rows_from_pages.restype = C.c_int
    lib.lbm_rows_from_pages.argtypes = [vp, vp, p(i32), p(i32), p(i32), i32, i32, vp, vp]
    lib.lbm_kv_append.restype = C.c_int
    lib.lbm_kv_append.argtypes = [vp, vp, i32, vp, i32, vp, i32, i32, i32, i32, vp]
    lib.lbm_qkv_prepare.restype = C.c_int
    lib.lbm_qkv_prepare.argtypes = [vp, i32, vp, vp, vp, vp, C.c_float, C.c_float, vp, i32, vp, vp, vp, i32, vp, vp, i32, i32, i32, i32, vp]
    lib.lbm_residual_norm.restype = C.c_int
    lib.lbm_residual_norm.argtypes = [vp, vp, i32, vp, vp, vp, C.c_float, vp, vp, i32, i32, vp]
    lib.lbm_linear.restype = C.c_int
    lib.lbm_linear.argtypes = [vp, vp, vp, vp, vp, vp, i32, i32, i32, i32, vp]
    lib.lbm_linear_norm.restype = C.c_int
    lib.lbm_linear_norm.argtypes = [vp, p(RowNorm), vp, vp, vp, vp, vp, vp, i32, i32, i32, i32, vp, C.c_size_t, vp]
    lib.lbm_linear_workspace_bytes.restype = C.c_size_t
    lib.lbm_linear_workspace_bytes.argtypes = [i32, i32, i32, i32]
    lib.lbm_linear_prefetch_hint.restype = C.c_int
    lib.lbm_linear_prefetch_hint.argtypes = [vp, C.c_size_t]
    lib.lbm_linear_stats_tiles.restype = i32
    lib.lbm_linear_stats_tiles.argtypes = [i32, i32]
    lib.lbm_qkv_linear_prepare_norm.restype = C.c_int
    lib.lbm_qkv_linear_prepare_norm.argtypes = [vp, p(RowNorm), vp, vp, i32, i32, vp, vp, vp, vp, C.c_float, C.c_float, vp, i32, vp, vp, vp, vp, vp, i32, i32, i32, vp]
    lib.lbm_qkv_linear_prepare.restype = C.c_int
    lib.lbm_qkv_linear_prepare.argtypes = [vp, vp, vp, i32, i32, vp, vp, vp, vp, C.c_float, C.c_float, vp, i32, vp, vp, vp, vp, vp, i32, i32, i32, vp]
    lib.lbm_attn_workspace_bytes.restype = C.c_size_t
    lib.lbm_attn_workspace_bytes.argtypes = [p(AttnStream), i32, i32, i32]
    lib.lbm_attn_run.restype = C.c_int
    lib.lbm_attn_run.argtypes = [vp, vp, vp, vp, vp, vp, p(AttnStream), i32, i32, i32, i32, i32,
                                 C.c_float, vp, C.c_size_t, vp]
    lib.lbm_attn_run_append.restype = C.c_int
    lib.lbm_attn_run_append.argtypes = [vp, vp, vp, vp, vp, vp, vp, i32, p(AttnStream), i32, i32, i32, i32, i32,
                                        C.c_float, vp, C.c_size_t, vp]
    lib.lbm_attn_run_call.restype = C.c_int
    lib.lbm_attn_run_call.argtypes = [C.c_char_p, vp]
    lib.lbm_attn_run_live.restype = C.c_int
    lib.lbm_attn_run_live.argtypes = [vp, vp, vp, vp, vp, vp, vp, p(AttnStream), i32, i32, i32, i32, i32,
                                      C.c_float, vp, C.c_size_t, vp]
    lib.lbm_attn_run_static.restype = C.c_int
    lib.lbm_attn_run_static.argtypes = [vp, vp, vp, vp, vp, vp, p(AttnStream), i32, i32, i32, i32, i32, C.c_float, vp]
    lib.lbm_block_scratch_bytes.restype = C.c_size_t
    lib.lbm_block_scratch_bytes.argtypes = [i32, i32, i32]
    lib.lbm_block_run.restype = C.c_int
    lib.lbm_block_run.argtypes = [p(BlockWeights), p(BlockCall), vp]
    lib.lbm_group_outputs.restype = C.c_int
    lib.lbm_group_outputs.argtypes = [p(vp), p(vp), i32, C.c_int64, C.c_int64, vp]
    lib.lbm_stream_table.restype = C.c_int
    lib.lbm_stream_table.argtypes = [vp, vp, C.c_int64, vp, i32, i32, i32, vp]
    lib.lbm_normalise_images.restype = C.c_int
    lib.lbm_normalise_images.argtypes = [vp, vp, vp, vp, i32, C.c_int64, C.c_int64, vp]
    lib.lbm_patch_tokens.restype = C.c_int
    lib.lbm_patch_tokens.argtypes = [vp, vp, vp, i32, i32, i32, vp]
    if lib.lbm_abi_version() != ABI_VERSION:
        raise RuntimeError(f"{LIB_PATH}: ABI version {lib.lbm_abi_version()}, binding expects {ABI_VERSION}")
    return lib


lib = _load()


def _load_host():
    """The extension module of the attention calls' host side (``csrc/host_calls.cpp``)."""
    if not os.path.exists(HOST_PATH):
        raise RuntimeError(f"{HOST_PATH} is not built; run `python -c 'import __graft_entry__ as g; g.build()'`")
    loader = importlib.machinery.ExtensionFileLoader("lbm_host", HOST_PATH)
    module = importlib.util.module_from_spec(importlib.util.spec_from_loader("lbm_host", loader))
    loader.exec_module(module)
    if getattr(module, "ABI_VERSION", None) != ABI_VERSION:
        raise RuntimeError(f"{HOST_PATH}: built for ABI version {getattr(module, 'ABI_VERSION', None)}, binding expects {ABI_VERSION}")
    return module


host = _load_host()


class LbmError(RuntimeError):
    pass


def check(rc: int) -> None:
    if rc != OK:
        msg = lib.lbm_last_error().decode("utf-8", "replace")
        if rc == ERR_INVALID:
            raise ValueError(msg)
        raise LbmError(f"lbm error {rc}: {msg}")


def q_scale_log2(sm_scale: float) -> float:
    """The ``q_scale`` to hand the producers so that ``lbm_attn_run`` can be called with
    ``sm_scale = 0``: the softmax scale times log2(e), as a float32 value."""
    return struct.unpack("f", struct.pack("f", sm_scale * 1.4426950408889634))[0]


def stream_handle(device) -> int:
    """The current HIP stream of ``device`` as an integer, which every ``void*`` argument of the
    binding takes.  One C call instead of building a ``torch.cuda.Stream`` object per launch (5 us
    each, several hundred per aggregator frame)."""
    import torch
    idx = device.index if getattr(device, "index", None) is not None else torch.cuda.current_device()
    return torch._C._cuda_getCurrentRawStream(idx)


def stream_ptr(device) -> C.c_void_p:
    """``stream_handle`` as a ``c_void_p``."""
    return C.c_void_p(stream_handle(device))
