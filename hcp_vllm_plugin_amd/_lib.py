"""ctypes binding of ``libhcp_mi355x.so`` (the C ABI in include/hcp_mi355x.h).

The library is built in-tree by ``hcp_vllm_plugin_amd.build`` (``__graft_entry__.build()``)
and loaded from this package directory.  Loading it after ``import torch`` makes
its ``libamdhip64.so.7`` dependency resolve to the HIP runtime torch already
loaded (same soname), so the raw ``hipStream_t`` of torch's current stream and
torch's device pointers are valid in the library.

There is no fallback: if the library is missing or fails to load, every entry
point raises ``RuntimeError``.
"""

from __future__ import annotations

import contextlib
import ctypes
import functools
import os
import threading
import time
from typing import NamedTuple

import torch  # noqa: F401  (must be loaded first: shares its HIP runtime)

LIB_NAME = "libhcp_mi355x.so"
LIB_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), LIB_NAME)

HCP_OK = 0
HCP_EINVAL = -1
HCP_EUNSUPPORTED = -2
HCP_ELAUNCH = -3
HCP_EWORKSPACE = -4

# include/hcp_mi355x.h HCP_NOALLOC_SCRATCH_BYTES
NOALLOC_SCRATCH_BYTES = 16 << 20

DTYPE_F16 = 0
DTYPE_BF16 = 1
DTYPE_F32 = 2
DTYPE_I32 = 3
DTYPE_I64 = 4

_STATUS_NAMES = {
    HCP_EINVAL: "EINVAL",
    HCP_EUNSUPPORTED: "EUNSUPPORTED",
    HCP_ELAUNCH: "ELAUNCH",
    HCP_EWORKSPACE: "EWORKSPACE",
}

# Every symbol include/hcp_mi355x.h declares.
EXPORTED_SYMBOLS = (
    "hcp_abi_version",
    "hcp_last_error",
    "hcp_attn_fwd_lse",
    "hcp_attn_fwd_lse_merge",
    "hcp_varlen_block_m",
    "hcp_plan_varlen_tiles",
    "hcp_attn_fwd_varlen",
    "hcp_attn_fwd_varlen_merge",
    "hcp_split_limits",
    "hcp_plan_fwd_split",
    "hcp_attn_fwd_lse_split",
    "hcp_plan_varlen_split",
    "hcp_varlen_launch",
    "hcp_fetch_metadata",
    "hcp_wait_metadata",
    "hcp_plan_decode_splits",
    "hcp_decode_workspace_bytes",
    "hcp_decode_splitkv",
    "hcp_plan_decode_lists",
    "hcp_decode_launch",
    "hcp_decode_paged_workspace",
    "hcp_decode_paged",
    "hcp_decode_splitkv_acc",
    "hcp_decode_splitkv_noalloc",
    "hcp_merge_attn_states",
    "hcp_reshape_and_cache",
    "hcp_gather_paged_kv",
)

ABI_VERSION = 11


class KvSegment(ctypes.Structure):
    """``hcp_kv_segment`` (include/hcp_mi355x.h)."""

    _fields_ = [
        ("k_addr", ctypes.c_uint64),
        ("v_addr", ctypes.c_uint64),
        ("block_table", ctypes.c_uint64),
        ("stride_tok", ctypes.c_int64),
        ("stride_head", ctypes.c_int64),
        ("stride_block", ctypes.c_int64),
        ("start", ctypes.c_int64),
        ("len", ctypes.c_int64),
        ("block_size", ctypes.c_int32),
        ("num_blocks", ctypes.c_int32),
    ]


class VarlenEntry(ctypes.Structure):
    """``hcp_varlen_entry`` (include/hcp_mi355x.h)."""

    _fields_ = [
        ("q_start", ctypes.c_int64),
        ("q_len", ctypes.c_int64),
        ("causal_offset", ctypes.c_int64),
        ("kv", KvSegment),
    ]


class PagedCacheDesc(ctypes.Structure):
    """``hcp_paged_cache`` (include/hcp_mi355x.h)."""

    _fields_ = [
        ("k_addr", ctypes.c_uint64),
        ("v_addr", ctypes.c_uint64),
        ("stride_block", ctypes.c_int64),
        ("stride_head", ctypes.c_int64),
        ("stride_tok", ctypes.c_int64),
        ("num_blocks", ctypes.c_int64),
        ("block_size", ctypes.c_int32),
        ("reserved", ctypes.c_int32),
    ]


class DecodeSplit(ctypes.Structure):
    """``hcp_decode_split`` (include/hcp_mi355x.h)."""

    _fields_ = [
        ("entry", ctypes.c_int32),
        ("key_begin", ctypes.c_int32),
        ("key_end", ctypes.c_int32),
        ("slot", ctypes.c_int32),
    ]


class DecodeArgs(ctypes.Structure):
    """``hcp_decode_args`` (include/hcp_mi355x.h)."""

    _fields_ = [
        ("q", ctypes.c_uint64),
        ("q_stride_tok", ctypes.c_int64),
        ("q_stride_head", ctypes.c_int64),
        ("works", ctypes.c_uint64),
        ("seq_partial_start", ctypes.c_uint64),
        ("seq_rows", ctypes.c_uint64),
        ("workspace", ctypes.c_uint64),
        ("workspace_bytes", ctypes.c_uint64),
        ("acc_o", ctypes.c_uint64),
        ("acc_stride_tok", ctypes.c_int64),
        ("acc_stride_head", ctypes.c_int64),
        ("acc_lse", ctypes.c_uint64),
        ("acc_lse_stride_head", ctypes.c_int64),
        ("out", ctypes.c_uint64),
        ("o_stride_tok", ctypes.c_int64),
        ("o_stride_head", ctypes.c_int64),
        ("lse", ctypes.c_uint64),
        ("lse_stride_head", ctypes.c_int64),
        ("kv_base", ctypes.c_uint64),
        ("num_works", ctypes.c_int32),
        ("num_wgs", ctypes.c_int32),
        ("num_seqs", ctypes.c_int32),
        ("num_heads", ctypes.c_int32),
        ("num_kv_heads", ctypes.c_int32),
        ("head_dim", ctypes.c_int32),
        ("dtype", ctypes.c_int32),
        ("use_scratch", ctypes.c_int32),
        ("scale", ctypes.c_float),
        ("keep_nan", ctypes.c_int32),
    ]


class VarlenArgs(ctypes.Structure):
    """``hcp_varlen_args`` (include/hcp_mi355x.h)."""

    _fields_ = [
        ("q", ctypes.c_uint64),
        ("q_stride_tok", ctypes.c_int64),
        ("q_stride_head", ctypes.c_int64),
        ("out", ctypes.c_uint64),
        ("o_stride_tok", ctypes.c_int64),
        ("o_stride_head", ctypes.c_int64),
        ("lse", ctypes.c_uint64),
        ("lse_stride_head", ctypes.c_int64),
        ("entries", ctypes.c_uint64),
        ("tiles", ctypes.c_uint64),
        ("units", ctypes.c_uint64),
        ("workspace", ctypes.c_uint64),
        ("workspace_bytes", ctypes.c_uint64),
        ("acc_o", ctypes.c_uint64),
        ("acc_stride_tok", ctypes.c_int64),
        ("acc_stride_head", ctypes.c_int64),
        ("acc_lse", ctypes.c_uint64),
        ("acc_lse_stride_head", ctypes.c_int64),
        ("kv_base", ctypes.c_uint64),
        ("num_entries", ctypes.c_int32),
        ("num_tiles", ctypes.c_int32),
        ("piece_tiles", ctypes.c_int32),
        ("num_units", ctypes.c_int32),
        ("num_slots", ctypes.c_int32),
        ("num_heads", ctypes.c_int32),
        ("num_kv_heads", ctypes.c_int32),
        ("head_dim", ctypes.c_int32),
        ("dtype", ctypes.c_int32),
        ("causal", ctypes.c_int32),
        ("window", ctypes.c_int32),
        ("paged", ctypes.c_int32),
        ("acc_is_prefix", ctypes.c_int32),
        ("scale", ctypes.c_float),
    ]


class DecodePagedArgs(ctypes.Structure):
    """``hcp_decode_paged_args`` (include/hcp_mi355x.h)."""

    _fields_ = [
        ("q", ctypes.c_uint64),
        ("q_stride_tok", ctypes.c_int64),
        ("q_stride_head", ctypes.c_int64),
        ("kv", KvSegment),
        ("block_table_stride", ctypes.c_int64),
        ("block_table_width", ctypes.c_int64),
        ("seq_lens", ctypes.c_uint64),
        ("workspace", ctypes.c_uint64),
        ("workspace_bytes", ctypes.c_uint64),
        ("out", ctypes.c_uint64),
        ("o_stride_tok", ctypes.c_int64),
        ("o_stride_head", ctypes.c_int64),
        ("lse", ctypes.c_uint64),
        ("lse_stride_head", ctypes.c_int64),
        ("lens_dtype", ctypes.c_int32),
        ("num_seqs", ctypes.c_int32),
        ("window", ctypes.c_int32),
        ("num_heads", ctypes.c_int32),
        ("num_kv_heads", ctypes.c_int32),
        ("head_dim", ctypes.c_int32),
        ("dtype", ctypes.c_int32),
        ("keep_nan", ctypes.c_int32),
        ("scale", ctypes.c_float),
    ]


# include/hcp_mi355x.h HCP_DECODE_PAGED_MAX_SEQS
DECODE_PAGED_MAX_SEQS = 1024

_lock = threading.Lock()
_lib = None

_P = ctypes.c_void_p
_I64 = ctypes.c_int64
_I32 = ctypes.c_int32
_F = ctypes.c_float


def _declare(lib: ctypes.CDLL) -> None:
    lib.hcp_abi_version.restype = ctypes.c_int
    lib.hcp_abi_version.argtypes = []
    lib.hcp_last_error.restype = ctypes.c_char_p
    lib.hcp_last_error.argtypes = []
    lib.hcp_attn_fwd_lse.restype = ctypes.c_int
    lib.hcp_attn_fwd_lse.argtypes = [
        _P, _P, _P, _P, _P, _I64, _I64, _I32, _I32, _I32,
        _I64, _I64, _I64, _I64, _I64, _I64, _I64, _I64, _I64,
        _F, _I32, _I64, _I32, _I32, _P,
    ]
    lib.hcp_attn_fwd_lse_merge.restype = ctypes.c_int
    lib.hcp_attn_fwd_lse_merge.argtypes = [
        _P, _P, _P, _P, _P, _I64, _I64, _I32, _I32, _I32,
        _I64, _I64, _I64, _I64, _I64, _I64, _I64, _I64, _I64,
        _F, _I32, _I64, _I32, _P, _I64, _I64, _P, _I64, _I32, _I32, _P,
    ]
    lib.hcp_varlen_block_m.restype = ctypes.c_int
    lib.hcp_varlen_block_m.argtypes = [_I32, _I32]
    lib.hcp_plan_varlen_tiles.restype = ctypes.c_int
    lib.hcp_plan_varlen_tiles.argtypes = [_P, _I32, _I32, _I32, _P, _I32]
    lib.hcp_attn_fwd_varlen.restype = ctypes.c_int
    lib.hcp_attn_fwd_varlen.argtypes = [
        _P, _I64, _I64, _P, _I64, _I64, _P, _I64,
        _P, _I32, _P, _I32, _I32, _I32, _I32, _F, _I32, _I32, _I32, _I32, _P,
    ]
    lib.hcp_attn_fwd_varlen_merge.restype = ctypes.c_int
    lib.hcp_attn_fwd_varlen_merge.argtypes = [
        _P, _I64, _I64, _P, _I64, _I64, _P, _I64,
        _P, _I32, _P, _I32, _I32, _I32, _I32, _F, _I32, _I32, _I32,
        _P, _I64, _I64, _P, _I64, _I32, _I32, _P,
    ]
    lib.hcp_split_limits.restype = ctypes.c_int
    lib.hcp_split_limits.argtypes = [_I32, _P, _P, _P, _P]
    lib.hcp_plan_fwd_split.restype = ctypes.c_int
    lib.hcp_plan_fwd_split.argtypes = [_I64, _I64, _I32, _I32, _I32, _I32, _I64, _I32, _P, _P]
    lib.hcp_attn_fwd_lse_split.restype = ctypes.c_int
    lib.hcp_attn_fwd_lse_split.argtypes = [
        _P, _P, _P, _P, _P, _I64, _I64, _I32, _I32, _I32,
        _I64, _I64, _I64, _I64, _I64, _I64, _I64, _I64, _I64,
        _F, _I32, _I64, _I32, _P, _I64, _I64, _P, _I64, _I32,
        _I32, _I32, _P, ctypes.c_size_t, _I32, _P,
    ]
    lib.hcp_plan_varlen_split.restype = ctypes.c_int
    lib.hcp_plan_varlen_split.argtypes = [
        _P, _I32, _I32, _I32, _I32, _I32, _I32, _P, _I32, _P, _P, _P, _P, _P,
    ]
    lib.hcp_varlen_launch.restype = ctypes.c_int
    lib.hcp_varlen_launch.argtypes = [_P, _P]
    lib.hcp_fetch_metadata.restype = ctypes.c_int
    lib.hcp_fetch_metadata.argtypes = [
        _P, _I32, _I64, _P, _I32, _I64, _P, _I32, _I64, _I32, _I64, _P, _I64, _P, _P,
    ]
    lib.hcp_wait_metadata.restype = ctypes.c_int
    lib.hcp_wait_metadata.argtypes = [_P, _I64, _P]
    lib.hcp_plan_decode_splits.restype = ctypes.c_int
    lib.hcp_plan_decode_splits.argtypes = [_P, _I32, _P, _I32, _I32, _I32, _P, _I32, _P]
    lib.hcp_decode_workspace_bytes.restype = ctypes.c_size_t
    lib.hcp_decode_workspace_bytes.argtypes = [_I32, _I32, _I32]
    lib.hcp_decode_splitkv.restype = ctypes.c_int
    lib.hcp_decode_splitkv.argtypes = [
        _P, _I64, _I64, _P, _I32, _P, _I32, _P, _I32, _P, ctypes.c_size_t,
        _P, _I64, _I64, _P, _I64, _I32, _I32, _I32, _F, _I32, _P,
    ]
    lib.hcp_plan_decode_lists.restype = ctypes.c_int
    lib.hcp_plan_decode_lists.argtypes = [
        _P, _I32, _P, _I32, _I32, _I32, _P, _P, _I32, _P, _P,
    ]
    lib.hcp_decode_launch.restype = ctypes.c_int
    lib.hcp_decode_launch.argtypes = [_P, _P]
    lib.hcp_decode_paged_workspace.restype = ctypes.c_size_t
    lib.hcp_decode_paged_workspace.argtypes = [_I32, _I32, _I32, _I32]
    lib.hcp_decode_paged.restype = ctypes.c_int
    lib.hcp_decode_paged.argtypes = [_P, _P]
    lib.hcp_decode_splitkv_acc.restype = ctypes.c_int
    lib.hcp_decode_splitkv_acc.argtypes = [
        _P, _I64, _I64, _P, _I32, _P, _I32, _P, _I32, _P, ctypes.c_size_t,
        _P, _I64, _I64, _P, _I64,
        _P, _I64, _I64, _P, _I64, _I32, _I32, _I32, _F, _I32, _P,
    ]
    lib.hcp_decode_splitkv_noalloc.restype = ctypes.c_int
    lib.hcp_decode_splitkv_noalloc.argtypes = [
        _P, _I64, _I64, _P, _I32, _P, _I32, _P, _I32,
        _P, _I64, _I64, _P, _I64, _I32, _I32, _I32, _F, _I32, _P,
    ]
    lib.hcp_reshape_and_cache.restype = ctypes.c_int
    lib.hcp_reshape_and_cache.argtypes = [
        _P, _I64, _I64, _P, _I64, _I64, _P, _I32, _I64, _I32, _I32, _P, _I32, _P,
    ]
    lib.hcp_gather_paged_kv.restype = ctypes.c_int
    lib.hcp_gather_paged_kv.argtypes = [_P, _I32, _P, _I64, _I32, _I32, _I32, _P, _P, _P]
    lib.hcp_merge_attn_states.restype = ctypes.c_int
    lib.hcp_merge_attn_states.argtypes = [
        _P, _I64, _I64, _I32, _P, _I64,
        _P, _I64, _I64, _I32, _P, _I64,
        _P, _I64, _I64, _I32, _P, _I64,
        _I64, _I32, _I32, _P,
    ]


def lib() -> ctypes.CDLL:
    """Load (once) and return the HIP library; raise if it is not built."""
    global _lib
    if _lib is not None:
        return _lib
    with _lock:
        if _lib is None:
            if not os.path.exists(LIB_PATH):
                raise RuntimeError(
                    f"{LIB_NAME} is not built ({LIB_PATH} missing); run "
                    "`python -c 'import __graft_entry__ as g; g.build()'` or "
                    "`python -m hcp_vllm_plugin_amd.build`"
                )
            try:
                handle = ctypes.CDLL(LIB_PATH, mode=ctypes.RTLD_LOCAL)
            except OSError as exc:
                raise RuntimeError(f"cannot load {LIB_PATH}: {exc}") from exc
            _declare(handle)
            ver = handle.hcp_abi_version()
            if ver != ABI_VERSION:
                raise RuntimeError(f"{LIB_NAME} ABI {ver}, expected {ABI_VERSION}")
            _lib = handle
    return _lib


def check(rc: int, what: str) -> None:
    """Turn a negative hcp_status into RuntimeError with the library's text."""
    if rc < 0:
        msg = lib().hcp_last_error().decode(errors="replace")
        raise RuntimeError(f"{what} failed ({_STATUS_NAMES.get(rc, rc)}): {msg}")


def dtype_code(dt: torch.dtype) -> int:
    if dt == torch.float16:
        return DTYPE_F16
    if dt == torch.bfloat16:
        return DTYPE_BF16
    if dt == torch.float32:
        return DTYPE_F32
    raise ValueError(f"unsupported dtype {dt}")


# the raw handle without building a torch.cuda.Stream around it, where this
# torch has the call
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def stream_ptr(device: torch.device) -> int:
    """Raw hipStream_t of torch's current stream on ``device``."""
    if _raw_stream is not None and device.index is not None:
        return _raw_stream(device.index)
    return torch.cuda.current_stream(device).cuda_stream


class SplitLimits(NamedTuple):
    """``hcp_split_limits`` (include/hcp_mi355x.h)."""

    max_units: int
    min_keys: int
    max_pieces: int
    max_workspace: int


@functools.lru_cache(maxsize=None)  # one entry per head_dim
def split_limits(head_dim: int) -> SplitLimits:
    if not 0 < head_dim <= 256:  # refused by the launch: nothing to cut
        return SplitLimits(0, 1 << 62, 0, 0)
    n = [ctypes.c_int32(0) for _ in range(3)]
    ws = ctypes.c_size_t(0)
    check(lib().hcp_split_limits(head_dim, *(ctypes.addressof(x) for x in n),
                                 ctypes.addressof(ws)), "hcp_split_limits")
    return SplitLimits(*(x.value for x in n), ws.value)


# per device: the last size there was no room for, and until when not to ask
# for as much again (a failed allocation empties torch's cache and waits for
# the device: not in every layer of every step)
_no_room: dict = {}
_NO_ROOM_S = 1.0


def scratch(nbytes: int, device: torch.device) -> torch.Tensor | None:
    """Stream-ordered scratch from torch's caching allocator for a launch that
    has another form without it; None when the device has no room for it."""
    held = _no_room.get(device.index)
    if held is not None:
        if time.monotonic() >= held[1]:
            _no_room.pop(device.index, None)
        elif nbytes >= held[0]:
            return None
    try:
        return torch.empty(nbytes, dtype=torch.uint8, device=device)
    except torch.OutOfMemoryError:
        _no_room[device.index] = (nbytes, time.monotonic() + _NO_ROOM_S)
        return None


_SAME_DEVICE = contextlib.nullcontext()


def on_device(device: torch.device):
    """``torch.cuda.device(device)``, without its two calls into the runtime
    when ``device`` is the current one already."""
    if device.index is None or device.index == torch.cuda.current_device():
        return _SAME_DEVICE
    return torch.cuda.device(device)
