"""Batched (varlen) prefill and split-KV decode on the HIP kernels.

The reference runs one flash launch per request and segment and gathers the
paged local KV into a contiguous copy first (ring_backend.py:611-832,
:617-624).  This module describes a whole batch as ``hcp_varlen_entry``
records -- query rows plus a KV segment that is either contiguous (staged
peer chunks) or paged (the local KV cache, read in place through the block
table) -- and runs one launch per segment kind:

* ``varlen_attn_with_lse``: causal (local) or non-causal (peer) prefill over
  every entry, tiles ordered longest-first by ``hcp_plan_varlen_tiles``.
* ``decode_attn``: split-KV decode of single-token queries; every segment of a
  sequence (peer and local) is split, and one reduce merges all partials.
* ``PagedDecode``: the same for a whole batch over one paged cache, without a
  plan: the kernel reads lengths and block tables itself.

Paged layouts the reference reads: vLLM 0.31 ``[nb, Hkv, bs, 2*D]`` with
K in ``[..., :D]`` and V in ``[..., D:]`` (file_connector.py:13-16,175-179),
and vLLM 0.23 ``[nb, 2, bs, Hkv, D]`` (ring_backend.py:601,617-624).
"""

from __future__ import annotations

import ctypes
import functools
from dataclasses import dataclass

import numpy as np

import torch

from . import _lib
from ._lib import KvSegment, VarlenEntry

__all__ = [
    "PagedCache",
    "segment_contiguous",
    "segment_paged",
    "varlen_attn_with_lse",
    "plan_varlen_tiles",
    "DecodeBatch",
    "PagedDecode",
    "decode_attn",
    "head_major",
]


@dataclass
class PagedCache:
    """A paged KV cache and its element strides.

    ``layout`` is ``"v031"`` for ``[nb, Hkv, bs, 2*D]`` or ``"v023"`` for
    ``[nb, 2, bs, Hkv, D]``; ``from_tensor`` infers it from the rank.
    """

    cache: torch.Tensor
    layout: str
    num_kv_heads: int
    head_dim: int
    block_size: int
    k_addr: int
    v_addr: int
    stride_tok: int
    stride_head: int
    stride_block: int

    @property
    def num_blocks(self) -> int:
        return int(self.cache.shape[0])

    @classmethod
    def from_tensor(cls, cache: torch.Tensor) -> "PagedCache":
        if cache.stride(-1) != 1:
            raise ValueError("paged cache: last dim must be contiguous")
        es = cache.element_size()
        if cache.dim() == 4:  # [nb, Hkv, bs, 2D]
            nb, hkv, bs, d2 = cache.shape
            d = d2 // 2
            return cls(cache, "v031", hkv, d, bs, cache.data_ptr(),
                       cache.data_ptr() + d * es,
                       cache.stride(2), cache.stride(1), cache.stride(0))
        if cache.dim() == 5 and cache.shape[1] == 2:  # [nb, 2, bs, Hkv, D]
            nb, _, bs, hkv, d = cache.shape
            return cls(cache, "v023", hkv, d, bs, cache.data_ptr(),
                       cache.data_ptr() + cache.stride(1) * es,
                       cache.stride(2), cache.stride(3), cache.stride(0))
        raise ValueError(f"unrecognised paged cache shape {tuple(cache.shape)}")


def segment_contiguous(k: torch.Tensor, v: torch.Tensor, start: int = 0,
                       length: int | None = None) -> KvSegment:
    """Segment over tokens ``[start, start+length)`` of k/v ``[T, Hkv, D]``."""
    if k.shape != v.shape or k.stride() != v.stride():
        raise ValueError("k and v must share shape and strides")
    _check_kv_layout(k.data_ptr(), v.data_ptr(), k.stride(0), k.stride(1), 0, k.element_size())
    if k.stride(-1) != 1:
        raise ValueError("k/v head_dim must be contiguous")
    n = k.shape[0] - start if length is None else length
    if start < 0 or n < 0 or start + n > k.shape[0]:
        raise ValueError("segment out of range")
    s = KvSegment()
    s.k_addr = k.data_ptr()
    s.v_addr = v.data_ptr()
    s.block_table = 0
    s.stride_tok = k.stride(0)
    s.stride_head = k.stride(1)
    s.stride_block = 0
    s.start = start
    s.len = n
    s.block_size = 0
    s._keep = (k, v)  # the descriptor holds raw addresses: keep the storage alive
    return s


def _check_kv_layout(k_addr: int, v_addr: int, stride_tok: int, stride_head: int,
                     stride_block: int, esize: int) -> None:
    """Kernel loadability: 16-byte aligned rows, token stride below 2^24 elements."""
    if k_addr % 16 or v_addr % 16:
        raise ValueError("k/v base addresses must be 16-byte aligned")
    if (stride_tok * esize) % 16 or (stride_head * esize) % 16 or (stride_block * esize) % 16:
        raise ValueError("k/v strides must be multiples of 16 bytes")
    if not 0 < stride_tok < (1 << 24):
        raise ValueError("k/v token stride must be in (0, 2^24) elements")


def segment_paged(pc: PagedCache, block_table_row: torch.Tensor, start: int,
                  length: int) -> KvSegment:
    """Segment over tokens ``[start, start+length)`` of one request's paged KV.

    ``block_table_row`` is the request's int32 block-table row on the device
    (contiguous); token x lives in block ``row[x // bs]`` at ``x % bs``.
    """
    if block_table_row.dtype != torch.int32 or block_table_row.stride(-1) != 1:
        raise ValueError("block table row must be contiguous int32")
    _check_kv_layout(pc.k_addr, pc.v_addr, pc.stride_tok, pc.stride_head, pc.stride_block,
                     pc.cache.element_size())
    if pc.block_size <= 0 or pc.block_size & (pc.block_size - 1):
        raise ValueError("block_size must be a power of two")
    if start < 0 or length < 0:
        raise ValueError("negative segment start/length")
    nblk = (start + length + pc.block_size - 1) // pc.block_size
    if length > 0 and nblk > block_table_row.shape[0]:
        raise ValueError("segment extends past the block-table row")
    s = KvSegment()
    s.k_addr = pc.k_addr
    s.v_addr = pc.v_addr
    s.block_table = block_table_row.data_ptr()
    s.stride_tok = pc.stride_tok
    s.stride_head = pc.stride_head
    s.stride_block = pc.stride_block
    s.start = start
    s.len = length
    s.block_size = pc.block_size
    s.num_blocks = pc.num_blocks if pc.num_blocks < (1 << 31) else 0
    s._keep = (pc.cache, block_table_row)  # raw addresses inside: keep them alive
    return s


def trim_segment(seg: KvSegment, skip: int) -> KvSegment:
    """The same keys without the first ``skip`` (0 <= skip <= len)."""
    if not 0 <= skip <= seg.len:
        raise ValueError("trim beyond the segment")
    s = KvSegment()
    ctypes.memmove(ctypes.addressof(s), ctypes.addressof(seg), ctypes.sizeof(KvSegment))
    s.start = seg.start + skip
    s.len = seg.len - skip
    s._keep = getattr(seg, "_keep", None)
    return s


def window_tail(segments: list, window: int | None) -> list:
    """The last ``window`` keys of the concatenation of ``segments`` (in
    order): what a query at the last position sees under a sliding window
    (ring_backend.py:397-398 with qpos = len - 1).  None keeps all keys."""
    segs = [s for s in segments if s is not None and s.len > 0]
    if window is None:
        return segs
    if window <= 0:
        raise ValueError("window must be a positive number of keys")
    out, need = [], window
    for s in reversed(segs):
        if need == 0:
            break
        out.append(s if s.len <= need else trim_segment(s, s.len - need))
        need -= min(need, s.len)
    return out[::-1]


def make_entry(q_start: int, q_len: int, seg: KvSegment, causal_offset: int = 0) -> VarlenEntry:
    e = VarlenEntry()
    e.q_start = q_start
    e.q_len = q_len
    e.causal_offset = causal_offset
    e.kv = seg
    e._keep = getattr(seg, "_keep", None)
    return e


def _nbytes_addr(a) -> tuple[int, int]:
    if isinstance(a, np.ndarray):
        return a.nbytes, a.ctypes.data
    return ctypes.sizeof(a), ctypes.addressof(a)


def _upload(arrays, device: torch.device):
    """Copy ctypes or numpy arrays to the device in one asynchronous copy from
    pinned memory on the current stream.

    Returns (device byte tensor, [address of each array on the device]), each
    array 256-byte aligned.  The pinned block comes from torch's caching host
    allocator, which keeps it until the copy has completed.
    """
    offs, total = [], 0
    for a in arrays:
        offs.append(total)
        total += (_nbytes_addr(a)[0] + 255) & ~255
    host = torch.empty(max(total, 256), dtype=torch.uint8, pin_memory=True)
    base = host.data_ptr()
    for a, o in zip(arrays, offs):
        nb, addr = _nbytes_addr(a)
        ctypes.memmove(base + o, addr, nb)
    dev = host.to(device, non_blocking=True)
    return dev, [dev.data_ptr() + o for o in offs]


# hcp_varlen_entry as a numpy record (include/hcp_mi355x.h), for building a
# whole batch's entries with array operations instead of one object each
ENTRY_DTYPE = np.dtype({
    "names": ["q_start", "q_len", "causal_offset", "k_addr", "v_addr", "block_table",
              "stride_tok", "stride_head", "stride_block", "start", "len", "block_size",
              "num_blocks"],
    "formats": ["<i8", "<i8", "<i8", "<u8", "<u8", "<u8", "<i8", "<i8", "<i8", "<i8", "<i8",
                "<i4", "<i4"],
    "offsets": [0, 8, 16, 24, 32, 40, 48, 56, 64, 72, 80, 88, 92],
    "itemsize": 96,
})
assert ENTRY_DTYPE.itemsize == ctypes.sizeof(VarlenEntry)

# hcp_decode_work: an entry and its split
WORK_DTYPE = np.dtype([("e", ENTRY_DTYPE)] + [(f, "<i4") for f in (
    "key_begin", "key_end", "slot", "next", "r0", "r1", "r2", "r3")])
assert WORK_DTYPE.itemsize == 128
_CHUNK_WORDS = np.array([ENTRY_DTYPE.fields[f][1] // 8 for f in (
    "k_addr", "v_addr", "stride_tok", "stride_head")])


def paged_entry_array(pc: "PagedCache", block_table: torch.Tensor, rows, q_start, q_len,
                      causal_offset, start, length, relative: bool = False) -> np.ndarray:
    """Entries over the paged cache for many requests at once: entry i covers
    query rows [q_start[i], +q_len[i]) and tokens [start[i], +length[i]) of
    block-table row rows[i].  ``block_table`` is the batch's contiguous int32
    table on the device; all checks are done once for the batch.  ``relative``:
    the K and V addresses relative to ``pc.k_addr``, for a launch given it as
    ``kv_base``."""
    if block_table.dtype != torch.int32 or not block_table.is_contiguous():
        raise ValueError("block table must be contiguous int32")
    _check_kv_layout(pc.k_addr, pc.v_addr, pc.stride_tok, pc.stride_head, pc.stride_block,
                     pc.cache.element_size())
    if pc.block_size <= 0 or pc.block_size & (pc.block_size - 1):
        raise ValueError("block_size must be a power of two")
    rows = np.asarray(rows, dtype=np.int64)
    start = np.asarray(start, dtype=np.int64)
    length = np.asarray(length, dtype=np.int64)
    if (start < 0).any() or (length < 0).any():
        raise ValueError("negative segment start/length")
    nblk = (start + length + pc.block_size - 1) // pc.block_size
    num_rows, width = block_table.shape
    # (as unsigned numbers: a negative row lies past the last one)
    past = rows.view(np.uint64) >= num_rows
    if ((length > 0) & ((nblk > width) | past)).any():
        if ((length > 0) & past).any():
            raise ValueError("the block table has no row for a request")
        raise ValueError("segment extends past the block-table row")
    a = np.zeros(len(rows), dtype=ENTRY_DTYPE)
    a["q_start"] = q_start
    a["q_len"] = q_len
    a["causal_offset"] = causal_offset
    a["k_addr"] = 0 if relative else pc.k_addr
    a["v_addr"] = pc.v_addr - pc.k_addr if relative else pc.v_addr
    a["block_table"] = block_table.data_ptr() + rows * block_table.stride(0) * 4
    a["stride_tok"] = pc.stride_tok
    a["stride_head"] = pc.stride_head
    a["stride_block"] = pc.stride_block
    a["start"] = start
    a["len"] = length
    a["block_size"] = pc.block_size
    a["num_blocks"] = pc.num_blocks if pc.num_blocks < (1 << 31) else 0
    return a


def plan_varlen_tiles(entries: list[VarlenEntry], causal: bool) -> list[tuple[int, int]]:
    """Host tile plan (entry, q_block), longest first (hcp_plan_varlen_tiles)."""
    L = _lib.lib()
    n = len(entries)
    arr = (VarlenEntry * max(n, 1))(*entries)
    bm = L.hcp_varlen_block_m(128, _lib.DTYPE_BF16)
    cap = sum((e.q_len + bm - 1) // bm for e in entries)
    tiles = (ctypes.c_int32 * max(2 * cap, 2))()
    rc = L.hcp_plan_varlen_tiles(ctypes.addressof(arr), n, int(causal), bm,
                                 ctypes.addressof(tiles), cap)
    _lib.check(rc, "hcp_plan_varlen_tiles")
    return [(tiles[2 * i], tiles[2 * i + 1]) for i in range(rc)]


# smallest block_size the paged prefill kernel reads in place (a wave's 16
# rows of a tile must lie in one block); smaller ones are gathered first
_MIN_PAGED_BLOCK = 16


@functools.lru_cache(maxsize=64)
def _varlen_cut(q_lens: bytes, kv_lens: bytes, offsets: bytes | None, window: int, heads):
    """(pieces, units, arguments) of the KV split of a launch with these sizes
    (int64 each; ``offsets`` None: not causal), None where it stays whole.  It
    follows from the sizes alone and takes 15 to 30 us of the host to find
    (known, 3 us), so the layers of a step share it."""
    n = len(q_lens) // 8
    ent = np.zeros(n, dtype=ENTRY_DTYPE)
    ent["q_len"], ent["len"] = np.frombuffer(q_lens, np.int64), np.frombuffer(kv_lens, np.int64)
    if offsets is not None:
        ent["causal_offset"] = np.frombuffer(offsets, np.int64)
    lim = _lib.split_limits(heads[2])
    if ent["len"].max() < lim.min_keys:
        return None
    ent["stride_tok"] = 1  # the real strides were checked with the tiles
    pieces, units = np.empty((2, lim.max_pieces, 4), dtype=np.int32)
    nu, ns, pt = (ctypes.c_int32(0) for _ in range(3))
    nbytes = ctypes.c_size_t(0)
    rc = _lib.lib().hcp_plan_varlen_split(
        ent.ctypes.data, n, int(offsets is not None), window, *heads, pieces.ctypes.data,
        lim.max_pieces, units.ctypes.data, ctypes.addressof(nu), ctypes.addressof(ns),
        ctypes.addressof(pt), ctypes.addressof(nbytes))
    _lib.check(rc, "hcp_plan_varlen_split")
    if rc == 0:
        return None
    pieces, units = pieces[:rc].copy(), units[:nu.value].copy()
    pieces.flags.writeable = units.flags.writeable = False  # shared by every launch of these sizes
    return pieces, units, {"key": (*heads, window), "pieces": rc, "units": nu.value,
                           "slots": ns.value, "piece_tiles": pt.value, "bytes": nbytes.value}


class VarlenLaunch:
    """A planned varlen launch: entries and tile list uploaded to the device.

    Build once per batch layout; ``run`` may be called repeatedly (e.g. per
    layer, or per benchmark step) with any q/out/lse of matching rows.  The
    plan is uploaded asynchronously on the current stream: run it on that
    stream (or synchronise first).
    """

    def __init__(self, entries, causal: bool, paged: bool, device: torch.device, keep=None,
                 heads: tuple[int, int, int] | None = None, window: int | None = None):
        """``entries``: a list of VarlenEntry, or an ENTRY_DTYPE array (then
        ``keep`` holds the tensors its addresses point into).

        ``heads = (num_heads, num_kv_heads, head_dim)`` and ``window`` of the
        runs to come let the plan cut long key ranges over few query rows into
        pieces (``hcp_plan_varlen_split``); a run with other values, or a plan
        built without them, takes the uncut launch."""
        L = _lib.lib()
        self.causal = bool(causal)
        self.paged = bool(paged)
        self.num_entries = len(entries)
        bm = L.hcp_varlen_block_m(128, _lib.DTYPE_BF16)
        if isinstance(entries, np.ndarray):
            if entries.dtype != ENTRY_DTYPE or not entries.flags.c_contiguous:
                raise ValueError("entry array must be contiguous ENTRY_DTYPE")
            if ((entries["block_table"] != 0) != self.paged).any():
                raise ValueError("all entries of a launch must share the KV form")
            arr = entries if self.num_entries else np.zeros(1, dtype=ENTRY_DTYPE)
            cap = int(((entries["q_len"] + bm - 1) // bm).sum())
            self._keep = keep
        else:
            for e in entries:
                if (e.kv.block_table != 0) != self.paged:
                    raise ValueError("all entries of a launch must share the KV form")
            arr = (VarlenEntry * max(self.num_entries, 1))(*entries)
            cap = sum((e.q_len + bm - 1) // bm for e in entries)
            # the entries point at K/V / cache / block-table storage by
            # address: hold those tensors for as long as this launch can run
            self._keep = [getattr(e, "_keep", None) for e in entries]
        # Paged prefill reads a wave's 16 rows of a tile from one block: over a
        # cache with shorter blocks the segments are gathered into one
        # contiguous K/V buffer on the device first (hcp_gather_paged_kv, one
        # launch per run), and the attention runs over that copy.
        self._gather = None
        if self.paged and self.num_entries:
            host = np.frombuffer(arr, dtype=ENTRY_DTYPE, count=self.num_entries).copy()
            if int(host["block_size"].min()) < _MIN_PAGED_BLOCK:
                lens = host["len"].astype(np.int64)
                out_start = np.zeros(self.num_entries, dtype=np.int64)
                out_start[1:] = np.cumsum(lens)[:-1]
                cont = host.copy()
                for f in ("block_table", "stride_block", "block_size", "num_blocks",
                          "k_addr", "v_addr"):
                    cont[f] = 0
                cont["start"] = out_start
                self._gather = {"paged": host, "out_start": out_start, "cont": cont,
                                "total": int(lens.sum()), "max_len": int(lens.max()),
                                "bufs": {}}
                arr = cont
                self.paged = False
        tiles = (ctypes.c_int32 * max(2 * cap, 2))()
        rc = L.hcp_plan_varlen_tiles(_nbytes_addr(arr)[1], self.num_entries,
                                     int(self.causal), bm, ctypes.addressof(tiles), cap)
        _lib.check(rc, "hcp_plan_varlen_tiles")
        self.num_tiles = rc
        split = self._plan_split(arr, heads, window)
        if self._gather is None:
            self._plan_dev, (self.entries_ptr, self.tiles_ptr, *sp) = _upload(
                [arr, tiles, *split], device)
        else:
            g = self._gather
            self._plan_dev, (g["paged_ptr"], g["start_ptr"], self.tiles_ptr, *sp) = _upload(
                [g["paged"], g["out_start"], tiles, *split], device)
            self.entries_ptr = None
        if split:
            self._split["ptrs"] = sp
        self.device = device

    def _plan_split(self, arr, heads, window):
        """The KV split of runs with these heads and window: records to upload
        ([pieces, units]), or [] for the uncut launch."""
        self._split = None
        if heads is None or not self.num_tiles or \
                self.num_tiles * heads[0] > _lib.split_limits(heads[2]).max_units:
            return []
        ent = np.frombuffer(arr, dtype=ENTRY_DTYPE, count=self.num_entries)
        win = int(window or 0) if self.causal else 0
        cut = _varlen_cut(ent["q_len"].tobytes(), ent["len"].tobytes(),
                          ent["causal_offset"].tobytes() if self.causal else None, win,
                          tuple(heads))
        if cut is None:
            return []
        pieces, units, self._split = cut[0], cut[1], dict(cut[2])
        return [pieces, units]

    def _gathered(self, q: torch.Tensor, num_kv_heads: int) -> int:
        """Gather mode: copy every entry's paged keys into a contiguous K/V
        buffer on the current stream; returns the device address of the
        entries over that buffer.

        The buffer (and its uploaded entries) is allocated on the first run
        of a (shape, stream) pair and reused by later runs on that stream,
        which the stream orders after each other; a run on another stream
        gets buffers of its own, so runs in flight on two streams never
        overwrite each other's keys.  Each buffer holds ``total * Hkv * D``
        16-bit elements of K and of V for as long as the launch lives."""
        g = self._gather
        head_dim = q.shape[2]
        st = torch.cuda.current_stream(q.device)
        key = (num_kv_heads, head_dim, q.dtype, st.cuda_stream)
        buf = g["bufs"].get(key)
        if buf is None:
            k = torch.empty(max(g["total"], 1), num_kv_heads, head_dim, dtype=q.dtype,
                            device=q.device)
            v = torch.empty_like(k)
            cont = g["cont"].copy()
            cont["k_addr"] = k.data_ptr()
            cont["v_addr"] = v.data_ptr()
            cont["stride_tok"] = num_kv_heads * head_dim
            cont["stride_head"] = head_dim
            cont_dev, (ptr,) = _upload([cont], q.device)
            buf = g["bufs"][key] = (k, v, cont_dev, ptr)
        k, v, _cont_dev, ptr = buf
        L = _lib.lib()
        rc = L.hcp_gather_paged_kv(g["paged_ptr"], self.num_entries, g["start_ptr"],
                                   g["max_len"], num_kv_heads, head_dim,
                                   _lib.dtype_code(q.dtype), k.data_ptr(),
                                   v.data_ptr(), _lib.stream_ptr(q.device))
        _lib.check(rc, "hcp_gather_paged_kv")
        return ptr

    def run(self, q: torch.Tensor, out: torch.Tensor, lse: torch.Tensor | None,
            num_kv_heads: int, scale: float, window: int | None = None,
            acc=None, acc_is_prefix: bool = True, kv_base: int = 0) -> None:
        """``window``: sliding window of a causal launch (query at p sees keys
        p - window < j <= p in its entry's frame); ignored when non-causal.

        ``acc=(o, lse)``: a partial state with out's rows, merged into the
        result in the same launch (``hcp_attn_fwd_varlen_merge``): with
        ``acc_is_prefix`` each row gets merge_attn_states(acc, this pass), the
        local pass taking the peer result as the prefix (ring_backend.py:354).
        ``lse`` may then be None; otherwise it receives the merged LSE.

        ``kv_base``: added to the addresses of paged entries (planned with
        addresses relative to a layer's cache)."""
        if self.num_tiles == 0:
            return
        if window is not None and window <= 0:
            raise ValueError("window must be a positive number of keys")
        if kv_base and self._gather is not None:
            raise ValueError("a gathering launch needs absolute cache addresses")
        num_heads, head_dim = q.shape[1], q.shape[2]
        win = int(window or 0) if self.causal else 0
        a = _lib.VarlenArgs()
        a.q, a.q_stride_tok, a.q_stride_head = q.data_ptr(), q.stride(0), q.stride(1)
        a.out, a.o_stride_tok, a.o_stride_head = out.data_ptr(), out.stride(0), out.stride(1)
        if lse is not None:
            a.lse, a.lse_stride_head = lse.data_ptr(), lse.stride(0)
        a.num_entries = self.num_entries
        a.num_heads, a.num_kv_heads, a.head_dim = num_heads, num_kv_heads, head_dim
        a.causal, a.window, a.paged = self.causal, win, self.paged
        a.scale, a.dtype, a.kv_base = float(scale), _lib.dtype_code(q.dtype), kv_base
        if acc is not None:
            a_o, a_lse = acc
            if a_o.dtype != q.dtype or a_o.stride(-1) != 1 or a_lse.dtype != torch.float32:
                raise ValueError("acc must be (out in q.dtype, float32 lse)")
            a.acc_o, a.acc_stride_tok, a.acc_stride_head = \
                a_o.data_ptr(), a_o.stride(0), a_o.stride(1)
            a.acc_lse, a.acc_lse_stride_head = a_lse.data_ptr(), a_lse.stride(0)
            a.acc_is_prefix = bool(acc_is_prefix)
        sp = self._split
        with _lib.on_device(q.device):
            a.entries = self.entries_ptr if self._gather is None else \
                self._gathered(q, num_kv_heads)
            # fp32 partials of a cut launch; without room for them it stays whole
            ws = None
            if sp is not None and sp["key"] == (num_heads, num_kv_heads, head_dim, win):
                ws = _lib.scratch(sp["bytes"], q.device)
            if ws is not None:
                a.workspace, a.workspace_bytes = ws.data_ptr(), sp["bytes"]
                a.tiles, a.num_tiles, a.piece_tiles = sp["ptrs"][0], sp["pieces"], sp["piece_tiles"]
                a.units, a.num_units, a.num_slots = sp["ptrs"][1], sp["units"], sp["slots"]
            else:
                a.tiles, a.num_tiles = self.tiles_ptr, self.num_tiles
            rc = _lib.lib().hcp_varlen_launch(ctypes.addressof(a), _lib.stream_ptr(q.device))
        _lib.check(rc, "hcp_varlen_launch")


def varlen_attn_with_lse(
    q: torch.Tensor,
    entries: list[VarlenEntry],
    causal: bool,
    num_kv_heads: int,
    scale: float,
    out: torch.Tensor | None = None,
    lse: torch.Tensor | None = None,
    window: int | None = None,
) -> tuple[torch.Tensor, torch.Tensor]:
    """One launch over all entries.  Rows not covered by an entry are left as
    given (``out``/``lse`` allocated here start as 0 / -inf).  ``window``: as
    ``VarlenLaunch.run``."""
    if q.dtype not in (torch.float16, torch.bfloat16) or q.stride(-1) != 1:
        raise ValueError("q must be float16/bfloat16 with contiguous head_dim")
    paged = bool(entries) and entries[0].kv.block_table != 0
    if out is None:
        out = torch.zeros_like(q, memory_format=torch.contiguous_format)
    if lse is None:
        lse = torch.full((q.shape[1], q.shape[0]), float("-inf"), dtype=torch.float32,
                         device=q.device)
    VarlenLaunch(entries, causal, paged, q.device, heads=(q.shape[1], num_kv_heads, q.shape[2]),
                 window=window).run(q, out, lse, num_kv_heads, scale, window)
    return out, lse


def head_major(t: torch.Tensor) -> torch.Tensor:
    """``t`` (``[n, Hkv, D]``) as an ``[n, Hkv, D]`` view of an ``[Hkv, n, D]``
    buffer, so each KV head's keys are one contiguous run (returned as is if
    already so stored)."""
    if t.dim() != 3 or t.stride() == (t.shape[2], t.shape[0] * t.shape[2], 1):
        return t
    return t.permute(1, 0, 2).contiguous().permute(1, 0, 2)


def head_chunks(num_heads: int, num_kv_heads: int) -> int:
    """Decode workgroups per (split, KV head): the split kernel takes up to 16
    query heads of a KV group at a time."""
    return -(-(num_heads // num_kv_heads) // 16)


def decode_workgroups(heads: int, num_cus: int = 256) -> int:
    """Workgroups of a decode launch per KV head and head chunk (``heads`` of
    them).  The split kernel runs one workgroup per CU (128 KB of LDS); its
    workgroups all get the same number of keys, so one round of the machine
    drains evenly."""
    return max(1, num_cus // heads)


class DecodeBatch:
    """A planned split-KV decode: entries and splits on the device (the fp32
    partials' workspace is taken per run).

    ``segments[s]`` lists the KV segments of sequence ``s`` (all keys visible
    to its single query, e.g. the staged peer prefix and the local paged KV
    including the current token).  The plan is uploaded asynchronously on the
    current stream: run it on that stream (or synchronise first).
    """

    def __init__(self, segments: list[list[KvSegment]], num_heads: int, num_kv_heads: int,
                 head_dim: int, device: torch.device, split_tokens: int | None = None,
                 rows: list[int] | None = None):
        """``rows``: the q / out / lse row of each sequence (default: its index)."""
        entries, seq_of = [], []
        for s, segs in enumerate(segments):
            for seg in segs:
                entries.append(make_entry(s if rows is None else rows[s], 1, seg, 0))
                seq_of.append(s)
        self.num_seqs = len(segments)
        self.num_entries = len(entries)
        self._contiguous = None
        n = max(self.num_entries, 1)
        arr = (VarlenEntry * n)(*entries)
        seq_arr = (ctypes.c_int32 * n)(*seq_of)
        self._plan(ctypes.addressof(arr), ctypes.addressof(seq_arr),
                   [e.kv.len for e in entries], num_heads, num_kv_heads, head_dim, split_tokens,
                   rows, device)
        # the segments point at K/V / cache / block-table storage by address
        self._keep = [getattr(e, "_keep", None) for e in entries]

    @classmethod
    def from_entries(cls, entries: np.ndarray, num_heads: int, num_kv_heads: int,
                     head_dim: int, device: torch.device, split_tokens: int | None = None,
                     keep=None, entry_seq: np.ndarray | None = None,
                     num_seqs: int | None = None, rows=None) -> "DecodeBatch":
        """Entries given as an ENTRY_DTYPE array; ``keep`` holds the tensors
        it points into.  By default one entry per sequence (sequence i = entry
        i = query row i); with ``entry_seq`` (int32, non-decreasing) entry j
        belongs to sequence ``entry_seq[j]`` of ``num_seqs`` -- a sequence's
        peer chunks and its local segment.  ``rows``: the out / lse row of
        each sequence (default: its index); the entries' q_start name the q rows."""
        if entries.dtype != ENTRY_DTYPE or not entries.flags.c_contiguous:
            raise ValueError("entry array must be contiguous ENTRY_DTYPE")
        self = cls.__new__(cls)
        n = len(entries)
        if entry_seq is None:
            seq_arr = np.arange(max(n, 1), dtype=np.int32)
            ns = n
        else:
            seq_arr = np.ascontiguousarray(entry_seq, dtype=np.int32)
            if len(seq_arr) != n or num_seqs is None:
                raise ValueError("entry_seq needs one sequence per entry and num_seqs")
            ns = int(num_seqs)
            if n == 0:
                seq_arr = np.zeros(1, dtype=np.int32)
        self.num_seqs = ns
        self.num_entries = n
        arr = entries if n else np.zeros(1, dtype=ENTRY_DTYPE)
        self._plan(arr.ctypes.data, seq_arr.ctypes.data, arr["len"][:n].tolist(), num_heads,
                   num_kv_heads, head_dim, split_tokens, rows, device)
        self._contiguous = entries["block_table"] == 0
        self._keep = keep
        return self

    def _plan(self, entries_addr, seq_addr, lens, num_heads, num_kv_heads, head_dim, split_tokens,
              rows, device) -> None:
        """Plan and upload: splits of at most ``split_tokens`` keys, one to a
        workgroup, or (None) an equal share of the batch's keys for every
        workgroup of the launch (``hcp_plan_decode_lists``)."""
        L = _lib.lib()
        n, ns = self.num_entries, self.num_seqs
        if rows is not None and len(rows) != ns:
            raise ValueError("rows needs one row per sequence")
        if split_tokens is None:
            wgs = decode_workgroups(num_kv_heads * head_chunks(num_heads, num_kv_heads))
            cap = n + wgs
        else:
            wgs = 0
            cap = sum(-(-x // split_tokens) for x in lens)
        self.split_tokens = split_tokens or max(1, -(-sum(lens) // wgs))  # keys to a workgroup
        # one block: partial starts, rows and records (uploaded), entry of each record
        rows_at = (4 * (ns + 1) + 255) & ~255
        works_at = rows_at + (0 if rows is None else (4 * ns + 255) & ~255)
        entry_at = works_at + 128 * max(cap, 1)
        block = np.empty(entry_at + 4 * max(cap, 1), dtype=np.uint8)
        base = block.ctypes.data
        if rows is not None:
            block[rows_at:rows_at + 4 * ns].view(np.int32)[:] = rows
        m = ctypes.c_int32(0)
        rc = L.hcp_plan_decode_lists(
            entries_addr, n, seq_addr, ns, wgs, split_tokens or 0, base + works_at,
            base + entry_at, cap, base, ctypes.addressof(m))
        _lib.check(rc, "hcp_plan_decode_lists")
        self.num_splits = rc
        self.num_heads = num_heads
        self.num_kv_heads = num_kv_heads
        self.head_dim = head_dim
        self.ws_bytes = int(L.hcp_decode_workspace_bytes(max(rc, 1), num_heads, head_dim))
        self.device = device
        # the records as words: copying those is one memcpy, copying records
        # goes field by field
        self._words = block[works_at:works_at + 128 * rc].view(np.uint64).reshape(rc, 16)
        self._work_entry = block[entry_at:entry_at + 4 * rc].view(np.int32)
        self._chunk_rows = None
        self._plan_dev, (dev,) = _upload([block[:works_at + 128 * max(rc, 1)]], device)
        a = self._args = _lib.DecodeArgs()
        a.works, a.num_works, a.num_wgs = dev + works_at, rc, m.value
        a.seq_partial_start, a.num_seqs = dev, ns
        a.seq_rows = 0 if rows is None else dev + rows_at
        a.workspace_bytes = self.ws_bytes
        a.num_heads, a.num_kv_heads, a.head_dim = num_heads, num_kv_heads, head_dim

    def rebind_chunks(self, rows: np.ndarray, keep=None) -> "DecodeBatch":
        """The same plan (splits, partial slots) over other chunks of the same
        lengths -- another layer's: row i of ``rows`` (uint64) is the K address,
        V address, token and head stride of the plan's i-th contiguous entry.
        Only the records go to the device (one small asynchronous copy)."""
        if self._contiguous is None:
            raise ValueError("rebind_chunks needs a plan made from an entry array")
        if self._chunk_rows is None:  # records of contiguous entries, and which of them
            which = np.cumsum(self._contiguous) - 1
            rec = np.nonzero(self._contiguous[self._work_entry])[0]
            self._chunk_rows = (rec, which[self._work_entry[rec]])
        if len(rows) != np.count_nonzero(self._contiguous):
            raise ValueError("rebind_chunks needs one row per contiguous entry")
        rec, src = self._chunk_rows
        words = self._words.copy()
        words[rec[:, None], _CHUNK_WORDS] = rows[src]
        other = object.__new__(type(self))
        other.__dict__.update(self.__dict__)
        other._words = words
        other._works_dev, (w_ptr,) = _upload([words], self.device)
        other._args = _lib.DecodeArgs.from_buffer_copy(self._args)
        other._args.works = w_ptr
        other._keep = keep
        return other

    def run(self, q: torch.Tensor, out: torch.Tensor, lse: torch.Tensor | None,
            scale: float, acc: tuple[torch.Tensor, torch.Tensor] | None = None,
            noalloc: bool = False, kv_base: int = 0, keep_nan: bool = False) -> None:
        """Decode into ``out`` (and ``lse``).  With ``acc = (o_acc [S, H, D] in
        q's dtype, lse_acc [H, S] float32)`` the accumulator is merged in by the
        same launch; ``out`` / ``lse`` may be the accumulator's own tensors.

        ``kv_base``: added to the addresses of paged segments (planned with
        addresses relative to a layer's cache).

        ``keep_nan``: a row whose scores hold a NaN comes out NaN, as from a
        prefill launch; otherwise the splits that hold one are left out.

        ``noalloc``: the partials live in the library's fixed per-GPU scratch
        (no workspace is taken, so nothing is allocated; calls overlapping on
        one GPU race).  Plans whose partials exceed
        ``_lib.NOALLOC_SCRATCH_BYTES`` raise."""
        L = _lib.lib()
        if noalloc and acc is not None:
            raise ValueError("noalloc decode has no accumulator form")
        a = _lib.DecodeArgs.from_buffer_copy(self._args)
        a.q, a.q_stride_tok, a.q_stride_head = q.data_ptr(), q.stride(0), q.stride(1)
        a.out, a.o_stride_tok, a.o_stride_head = out.data_ptr(), out.stride(0), out.stride(1)
        if lse is not None:
            a.lse, a.lse_stride_head = lse.data_ptr(), lse.stride(0)
        a.scale, a.dtype, a.kv_base = float(scale), _lib.dtype_code(q.dtype), kv_base
        a.keep_nan = keep_nan
        if acc is not None:
            ao, al = acc
            if ao.dtype != q.dtype or tuple(ao.shape) != tuple(q.shape) or ao.stride(-1) != 1:
                raise ValueError("acc o must match q's dtype and shape, contiguous head_dim")
            if al.dtype != torch.float32 or tuple(al.shape) != (q.shape[1], q.shape[0]) \
                    or al.stride(1) != 1:
                raise ValueError("acc lse must be float32 [H, S], contiguous along S")
            if not (ao.is_cuda and al.is_cuda):
                raise ValueError("accumulator must be on the GPU")
            a.acc_o, a.acc_stride_tok, a.acc_stride_head = ao.data_ptr(), ao.stride(0), ao.stride(1)
            a.acc_lse, a.acc_lse_stride_head = al.data_ptr(), al.stride(0)
        with _lib.on_device(q.device):
            if noalloc:
                a.use_scratch = 1
            else:
                # fp32 partials: stream-ordered scratch from torch's caching allocator
                ws = torch.empty(self.ws_bytes, dtype=torch.uint8, device=q.device)
                a.workspace = ws.data_ptr()
            rc = L.hcp_decode_launch(ctypes.addressof(a), _lib.stream_ptr(q.device))
        _lib.check(rc, "hcp_decode_launch")


class PagedDecode:
    """A pure decode batch over one paged cache, without a plan
    (``hcp_decode_paged``): query row r attends to the first ``seq_lens[r]``
    keys of row r of ``block_table`` (the last ``window`` of them).  Lengths
    and block ids are read on the device when a run executes; a length past its
    table row counts as the row's keys, so a caller that refuses such a batch
    checks the lengths itself.  One object serves every layer whose cache has
    ``pc``'s layout."""

    def __init__(self, pc: PagedCache, block_table: torch.Tensor, seq_lens: torch.Tensor,
                 num_heads: int, window: int | None):
        if block_table.dtype != torch.int32 or block_table.stride(-1) != 1:
            raise ValueError("block table must be int32 with contiguous rows")
        _check_kv_layout(pc.k_addr, pc.v_addr, pc.stride_tok, pc.stride_head, pc.stride_block,
                         pc.cache.element_size())
        if pc.block_size <= 0 or pc.block_size & (pc.block_size - 1):
            raise ValueError("block_size must be a power of two")
        n = seq_lens.shape[0]
        if block_table.dim() != 2 or block_table.shape[0] < n:
            raise ValueError("the block table has no row for a request")
        a = self._args = _lib.DecodePagedArgs()
        a.kv.block_table = block_table.data_ptr()
        a.kv.stride_tok, a.kv.stride_head = pc.stride_tok, pc.stride_head
        a.kv.stride_block, a.kv.block_size = pc.stride_block, pc.block_size
        a.kv.num_blocks = pc.num_blocks if pc.num_blocks < (1 << 31) else 0
        a.block_table_stride, a.block_table_width = block_table.stride(0), block_table.shape[1]
        a.seq_lens = seq_lens.data_ptr()
        a.lens_dtype = _lib.DTYPE_I64 if seq_lens.dtype == torch.int64 else _lib.DTYPE_I32
        a.num_seqs, a.window = n, int(window or 0)
        a.num_heads, a.num_kv_heads, a.head_dim = num_heads, pc.num_kv_heads, pc.head_dim
        a.workspace_bytes = _lib.lib().hcp_decode_paged_workspace(n, num_heads, pc.num_kv_heads,
                                                                  pc.head_dim)
        self._keep = (block_table, seq_lens)

    @staticmethod
    def takes(block_table: torch.Tensor, seq_lens: torch.Tensor, block_size: int) -> bool:
        """Whether a batch of this shape runs without a plan."""
        n = seq_lens.shape[0]
        if block_table.dim() != 2 or block_table.shape[0] < n:
            return False
        width = block_table.shape[1]
        return (0 < n <= _lib.DECODE_PAGED_MAX_SEQS and width > 0 and block_table.is_cuda
                and block_table.dtype == torch.int32 and block_table.stride(1) == 1
                and seq_lens.is_cuda and seq_lens.dim() == 1 and seq_lens.stride(0) == 1
                and seq_lens.dtype in (torch.int32, torch.int64)
                and width * block_size < 1 << 31 and width <= ((1 << 34) // block_size) // n)

    def run(self, q: torch.Tensor, out: torch.Tensor, pc: PagedCache, scale: float,
            keep_nan: bool = False) -> None:
        """One layer: its q, out and cache.  ``keep_nan``: as ``DecodeBatch.run``."""
        a = _lib.DecodePagedArgs.from_buffer_copy(self._args)
        a.q, a.q_stride_tok, a.q_stride_head = q.data_ptr(), q.stride(0), q.stride(1)
        a.out, a.o_stride_tok, a.o_stride_head = out.data_ptr(), out.stride(0), out.stride(1)
        a.kv.k_addr, a.kv.v_addr = pc.k_addr, pc.v_addr
        a.scale, a.dtype, a.keep_nan = float(scale), _lib.dtype_code(q.dtype), keep_nan
        with _lib.on_device(q.device):
            # fp32 partials: stream-ordered scratch from torch's caching allocator
            ws = torch.empty(a.workspace_bytes, dtype=torch.uint8, device=q.device)
            a.workspace = ws.data_ptr()
            rc = _lib.lib().hcp_decode_paged(ctypes.addressof(a), _lib.stream_ptr(q.device))
        _lib.check(rc, "hcp_decode_paged")


def decode_attn(
    q: torch.Tensor,
    segments: list[list[KvSegment]],
    num_kv_heads: int,
    scale: float,
    out: torch.Tensor | None = None,
    with_lse: bool = False,
    split_tokens: int | None = None,
    acc: tuple[torch.Tensor, torch.Tensor] | None = None,
):
    """Split-KV decode: q ``[S, H, D]`` (one token per sequence) over all
    segments of each sequence, merged (and merged into ``acc`` when given).
    Returns out (and lse ``[H, S]``)."""
    if q.dtype not in (torch.float16, torch.bfloat16) or q.stride(-1) != 1:
        raise ValueError("q must be float16/bfloat16 with contiguous head_dim")
    if len(segments) != q.shape[0]:
        raise ValueError("one segment list per query row")
    s, h, d = q.shape
    batch = DecodeBatch(segments, h, num_kv_heads, d, q.device, split_tokens)
    if out is None:
        out = torch.empty_like(q, memory_format=torch.contiguous_format)
    lse = torch.empty((h, s), dtype=torch.float32, device=q.device) if with_lse else None
    batch.run(q, out, lse, scale, acc)
    return (out, lse) if with_lse else out
