"""The C entries that the Python layer does not call, called as a C program
does: plans made by the library's planners, descriptors copied to the device,
plain arguments.  ``hcp_decode_splitkv``, ``_acc`` and ``_noalloc`` on splits of
``hcp_plan_decode_splits`` (an entry index and a key range each), and
``hcp_attn_fwd_varlen`` and ``_merge`` on tiles of ``hcp_plan_varlen_tiles``:
against the oracle, and against the launches with one argument block."""

import ctypes

import numpy as np
import pytest
import torch

from hcp_vllm_plugin_amd import _lib, merge_attn_states
from hcp_vllm_plugin_amd.varlen import (ENTRY_DTYPE, DecodeBatch, PagedCache, VarlenLaunch, _upload,
                                        make_entry, segment_contiguous, segment_paged)
from oracle import ring_oracle as orc
from tests._util import LSE_TOL, OUT_TOL, max_err, randn, scale_for

pytestmark = pytest.mark.gpu

SPLIT = np.dtype([("entry", "<i4"), ("key_begin", "<i4"), ("key_end", "<i4"), ("slot", "<i4")])


def _inputs(dev, seqs, h, hkv, d, dtype, seed):
    """Contiguous and paged segments of each (peer, local) pair of lengths,
    their keys and values, and one query row each."""
    gen = torch.Generator().manual_seed(seed)
    blocks = [-(-loc // 16) for _, loc in seqs]
    cache = randn(gen, (sum(blocks) + 2, hkv, 16, 2 * d), dtype)
    ids = torch.randperm(sum(blocks) + 2, generator=gen).to(torch.int32)
    bt = torch.zeros(len(seqs), max(blocks + [1]), dtype=torch.int32)
    at = 0
    for r, n in enumerate(blocks):
        bt[r, :n] = ids[at:at + n]
        at += n
    peers = [(randn(gen, (p, hkv, d), dtype), randn(gen, (p, hkv, d), dtype)) for p, _ in seqs]
    q = randn(gen, (len(seqs), h, d), dtype)
    cd, btd = cache.to(dev), bt.to(dev)
    pd = [(k.to(dev), v.to(dev)) for k, v in peers]
    pc, segs, kv = PagedCache.from_tensor(cd), [], []
    for r, (p, loc) in enumerate(seqs):
        segs.append(([segment_contiguous(*pd[r])] if p else [])
                    + ([segment_paged(pc, btd[r], 0, loc)] if loc else []))
        kl, vl = orc.gather_paged(cache.float(), bt[r], 0, loc, "v031")
        kv.append((torch.cat([peers[r][0].float(), kl]), torch.cat([peers[r][1].float(), vl])))
    return q, segs, kv, (cd, btd, pd)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("h,hkv,d", [(28, 4, 128), (6, 3, 64), (36, 2, 80), (4, 2, 256)])
@pytest.mark.parametrize("split", [64, 500])
def test_decode_entries(dev, dtype, h, hkv, d, split):
    seqs = [(700, 33), (0, 900), (65, 0), (0, 0), (1300, 1)]
    q, segs, kv, keep = _inputs(dev, seqs, h, hkv, d, dtype, d + split)
    L, n = _lib.lib(), len(seqs)
    entries, of = [], []
    for s, ss in enumerate(segs):
        for seg in ss:
            entries.append(make_entry(s, 1, seg, 0))
            of.append(s)
    arr = (_lib.VarlenEntry * len(entries))(*entries)
    seq = np.asarray(of, np.int32)
    cap = sum(-(-e.kv.len // split) for e in entries)
    splits, starts = np.zeros(cap, SPLIT), np.zeros(n + 1, np.int32)
    rc = L.hcp_plan_decode_splits(ctypes.addressof(arr), len(entries), seq.ctypes.data, n, 0, split,
                                  splits.ctypes.data, cap, starts.ctypes.data)
    _lib.check(rc, "hcp_plan_decode_splits")
    assert rc == cap == starts[-1]
    plan, (e_ptr, s_ptr, st_ptr) = _upload([arr, splits, starts], dev)
    scale, qd = scale_for(d), q.to(dev)
    nbytes = L.hcp_decode_workspace_bytes(rc, h, d)
    assert nbytes <= _lib.NOALLOC_SCRATCH_BYTES
    ws = torch.full((nbytes // 4,), float("nan"), device=dev)
    head = (qd.data_ptr(), qd.stride(0), qd.stride(1), e_ptr, len(entries), s_ptr, rc, st_ptr, n)
    tail = (h, hkv, d, scale, _lib.dtype_code(dtype), _lib.stream_ptr(dev))

    def fresh():
        return torch.full_like(qd, 7.0), torch.full((h, n), 7.0, device=dev)

    def outs(o, l):
        return (o.data_ptr(), o.stride(0), o.stride(1), l.data_ptr(), l.stride(0))

    out, lse = fresh()
    _lib.check(L.hcp_decode_splitkv(*head, ws.data_ptr(), nbytes, *outs(out, lse), *tail), "plain")
    fixed, fixed_l = fresh()
    _lib.check(L.hcp_decode_splitkv_noalloc(*head, *outs(fixed, fixed_l), *tail), "noalloc")
    acc_o = randn(torch.Generator().manual_seed(1), (n, h, d), dtype).to(dev)
    acc_l = torch.linspace(-3, 9, h * n, device=dev).view(h, n).contiguous()
    acc_l[0, :] = float("-inf")
    merged, merged_l = fresh()
    _lib.check(L.hcp_decode_splitkv_acc(*head, ws.data_ptr(), nbytes, acc_o.data_ptr(),
                                        acc_o.stride(0), acc_o.stride(1), acc_l.data_ptr(),
                                        acc_l.stride(0), *outs(merged, merged_l), *tail), "acc")
    batch = DecodeBatch(segs, h, hkv, d, dev, split_tokens=split)
    one, one_l = fresh()
    batch.run(qd, one, one_l, scale)
    both, both_l = fresh()
    batch.run(qd, both, both_l, scale, acc=(acc_o, acc_l))
    torch.cuda.synchronize()
    # the same pieces in the same slots: the same bits
    for a, b in ((out, fixed), (lse, fixed_l), (out, one), (lse, one_l), (merged, both),
                 (merged_l, both_l)):
        assert torch.equal(a, b)
    for r, (k, v) in enumerate(kv):
        o, l = orc.attn_with_lse(q[r:r + 1].float(), k, v, scale, None)
        tol = OUT_TOL[dtype] * max(1.0, o.abs().max().item() / 4)
        assert max_err(out[r:r + 1], o) <= tol
        assert max_err(lse[:, r:r + 1], l) <= LSE_TOL
        ml = torch.logaddexp(l, acc_l[:, r:r + 1].cpu())
        w, wa = torch.exp(l - ml).nan_to_num(0), torch.exp(acc_l[:, r:r + 1].cpu() - ml).nan_to_num(0)
        m = o * w.t()[..., None] + acc_o[r:r + 1].float().cpu() * wa.t()[..., None]
        assert max_err(merged[r:r + 1], m) <= max(tol, OUT_TOL[dtype] * m.abs().max().item() / 2)
        assert max_err(merged_l[:, r:r + 1], ml) <= LSE_TOL
    del keep, plan


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("h,hkv,d", [(8, 2, 128), (4, 2, 64), (4, 2, 256)])
@pytest.mark.parametrize("causal,window,paged", [(1, 0, 1), (1, 100, 1), (0, 0, 0), (1, 0, 0)])
def test_varlen_entries(dev, dtype, h, hkv, d, causal, window, paged):
    reqs = [(200, 700), (1, 40), (0, 64), (129, 129)]
    _, segs, kv, keep = _inputs(dev, [(0, n) if paged else (n, 0) for _, n in reqs], h, hkv, d,
                                dtype, d + window)
    rows = sum(t for t, _ in reqs)
    q = randn(torch.Generator().manual_seed(5), (rows, h, d), dtype)
    entries, at = [], 0
    for (t, n), (seg,) in zip(reqs, segs):
        entries.append(make_entry(at, t, seg, n - t if causal else 0))
        at += t
    L, n = _lib.lib(), len(entries)
    arr = (_lib.VarlenEntry * n)(*entries)
    bm = L.hcp_varlen_block_m(d, _lib.dtype_code(dtype))
    cap = sum(-(-t // bm) for t, _ in reqs)
    tiles = np.zeros((cap, 2), np.int32)
    rc = L.hcp_plan_varlen_tiles(ctypes.addressof(arr), n, causal, bm, tiles.ctypes.data, cap)
    assert rc == cap
    plan, (e_ptr, t_ptr) = _upload([arr, tiles], dev)
    scale, qd = scale_for(d), q.to(dev)
    out, lse = torch.full_like(qd, 7.0), torch.full((h, rows), 7.0, device=dev)
    head = (qd.data_ptr(), qd.stride(0), qd.stride(1))
    mid = (e_ptr, n, t_ptr, rc, h, hkv, d, scale, causal, window, paged)
    end = (_lib.dtype_code(dtype), _lib.stream_ptr(dev))
    _lib.check(L.hcp_attn_fwd_varlen(*head, out.data_ptr(), out.stride(0), out.stride(1),
                                     lse.data_ptr(), lse.stride(0), *mid, *end), "varlen")
    acc_o = randn(torch.Generator().manual_seed(6), (rows, h, d), dtype).to(dev)
    acc_l = torch.linspace(-2, 8, h * rows, device=dev).view(h, rows).contiguous()
    got, got_l = torch.full_like(qd, 7.0), torch.full_like(lse, 7.0)
    _lib.check(L.hcp_attn_fwd_varlen_merge(
        *head, got.data_ptr(), got.stride(0), got.stride(1), got_l.data_ptr(), got_l.stride(0),
        *mid, acc_o.data_ptr(), acc_o.stride(0), acc_o.stride(1), acc_l.data_ptr(),
        acc_l.stride(0), 1, *end), "varlen merge")
    one, one_l = torch.full_like(qd, 7.0), torch.full_like(lse, 7.0)
    VarlenLaunch(entries, bool(causal), bool(paged), dev).run(qd, one, one_l, hkv, scale,
                                                              window or None)
    want, want_l = torch.empty_like(qd), torch.empty_like(lse)
    merge_attn_states(want, acc_o, acc_l, out, lse, want_l)
    torch.cuda.synchronize()
    assert torch.equal(out, one) and torch.equal(lse, one_l)
    assert torch.equal(got, want) and torch.equal(got_l, want_l)
    at = 0
    for (t, nk), (k, v) in zip(reqs, kv):
        if t:
            o, l = orc.attn_with_lse(q[at:at + t].float(), k, v, scale,
                                     nk - t if causal else None, window or None)
            assert max_err(out[at:at + t], o) <= OUT_TOL[dtype] * max(1.0, o.abs().max().item() / 4)
            assert max_err(lse[:, at:at + t], l) <= LSE_TOL
        at += t
    assert ENTRY_DTYPE.itemsize == ctypes.sizeof(_lib.VarlenEntry)
    del keep, plan
