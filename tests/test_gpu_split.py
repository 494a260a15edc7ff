"""KV-split prefill against the oracle: pieces of one tile, ragged last tiles,
blocks left whole, rows a piece shows no key, windows, paged segments that
start inside a block, and the merge with a partial state (bit for bit the
split pass followed by ``merge_attn_states``).

The tolerances are the unsplit passes': the partials are f32, so a split adds
only the f32 rounding of the merge.
"""

import pytest
import torch

from hcp_vllm_plugin_amd import _lib, merge_attn_states, ring_attn_merged, ring_attn_with_lse
from hcp_vllm_plugin_amd.varlen import PagedCache, make_entry, segment_contiguous, segment_paged, \
    varlen_attn_with_lse
from oracle import ring_oracle as orc
from tests._util import LSE_TOL, OUT_TOL, max_err, outlier_k, randn, scale_for

pytestmark = pytest.mark.gpu


def _qkv(seed, tq, tk, h, hkv, d, dtype):
    gen = torch.Generator().manual_seed(seed)
    return (randn(gen, (tq, h, d), dtype),
            outlier_k(randn(gen, (tk, hkv, d), torch.float32), gen).to(dtype),
            randn(gen, (tk, hkv, d), dtype))


def _split(q, k, v, scale, off, window, piece, whole, acc=None):
    tq, h, d = q.shape
    out, lse = torch.full_like(q, 7.0), torch.full((h, tq), 7.0, device=q.device)
    dw = 64 if d <= 64 else 128 if d <= 128 else 256
    blocks, tiles = -(-tq // 128), -(-max(k.shape[0], 1) // 64)
    ws = torch.full(((blocks - whole) * -(-tiles // piece) * h * 128 * (dw + 1),), float("nan"),
                    device=q.device)
    a = (0, 0, 0, 0, 0, 0) if acc is None else (
        acc[0].data_ptr(), acc[0].stride(0), acc[0].stride(1), acc[1].data_ptr(),
        acc[1].stride(0), 1)
    L = _lib.lib()
    rc = L.hcp_attn_fwd_lse_split(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), lse.data_ptr(), tq, k.shape[0],
        h, k.shape[1], d, q.stride(0), q.stride(1), k.stride(0), k.stride(1), v.stride(0),
        v.stride(1), out.stride(0), out.stride(1), lse.stride(0), scale,
        0 if off is None else 1, off or 0, window or 0, *a, piece, whole, ws.data_ptr(),
        ws.numel() * 4, _lib.dtype_code(q.dtype), _lib.stream_ptr(q.device))
    _lib.check(rc, "hcp_attn_fwd_lse_split")
    torch.cuda.synchronize()
    return out, lse


# (tq, tk, causal offset or None, window, tiles per piece, blocks left whole)
CASES = [
    (1, 65, None, 0, 1, 0),        # one row, a piece of one key
    (33, 1000, 967, 0, 1, 0),      # one-tile pieces, ragged last tile
    (128, 512, None, 0, 3, 0),     # 8 tiles in 3 pieces (2, 3, 3)
    (257, 700, 443, 0, 2, 0),      # three blocks, the last of one row
    (257, 700, 443, 0, 2, 2),      # ... two of them whole
    (300, 300, 0, 0, 1, 0),        # diagonal: late pieces hidden from early rows
    (200, 900, 700, 150, 2, 0),    # window: rows with nothing in a piece
    (140, 300, -60, 0, 1, 0),      # leading rows see no key at all
    (130, 640, 510, 0, 100, 0),    # piece longer than the keys: nothing is cut
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("h,hkv,d", [(8, 2, 128), (4, 2, 64), (4, 4, 256), (6, 3, 80)])
@pytest.mark.parametrize("tq,tk,off,window,piece,whole", CASES)
def test_split_matches_oracle(dev, dtype, h, hkv, d, tq, tk, off, window, piece, whole):
    q, k, v = _qkv(tq + tk + d, tq, tk, h, hkv, d, dtype)
    scale = scale_for(d)
    qd, kd, vd = q.to(dev), k.to(dev), v.to(dev)
    out, lse = _split(qd, kd, vd, scale, off, window, piece, whole)
    o_ref, l_ref = orc.attn_with_lse(q, k, v, scale, off, window or None)
    seen = torch.isfinite(l_ref)
    assert torch.equal(torch.isfinite(lse.cpu()), seen)
    assert max_err(out, o_ref) <= OUT_TOL[dtype]
    assert max_err(lse.cpu()[seen], l_ref[seen]) <= LSE_TOL
    # merged with a partial state: the same as the pass and the merge after it
    acc_o, acc_l = out.flip(0).contiguous(), lse.flip(1).contiguous()
    got, got_l = _split(qd, kd, vd, scale, off, window, piece, whole, (acc_o, acc_l))
    want, want_l = torch.empty_like(out), torch.empty_like(lse)
    merge_attn_states(want, acc_o, acc_l, out, lse, want_l)
    assert torch.equal(got, want) and torch.equal(got_l, want_l)


@pytest.mark.parametrize("layout", ["v031", "v023"])
@pytest.mark.parametrize("new,keys,start", [(16, 8000, 0), (200, 9000, 7), (130, 12000, 40)])
def test_planned_split_of_a_paged_chunk(dev, layout, new, keys, start):
    """A chunk the planner cuts, read through the block table from a start
    inside a block: against the oracle and against the contiguous entry point
    (which plans its own cut)."""
    h, hkv, d, bs = 14, 2, 64, 16
    q, k, v = _qkv(new + keys, new, keys, h, hkv, d, torch.bfloat16)
    nb = -(-(start + keys) // bs)
    gen = torch.Generator().manual_seed(3)
    table = torch.randperm(nb + 3, generator=gen)[:nb].to(torch.int32)
    shape = (nb + 3, hkv, bs, 2 * d) if layout == "v031" else (nb + 3, 2, bs, hkv, d)
    cache = torch.full(shape, float("nan"), dtype=torch.bfloat16)
    pos = torch.arange(start, start + keys)
    blk, at = table.long()[pos // bs], pos % bs
    if layout == "v031":
        cache[blk, :, at, :d], cache[blk, :, at, d:] = k, v
    else:
        cache[blk, 0, at], cache[blk, 1, at] = k, v
    cache, table, qd = cache.to(dev), table.to(dev), q.to(dev)
    ent = [make_entry(0, new, segment_paged(PagedCache.from_tensor(cache), table, start, keys),
                      keys - new)]
    scale = scale_for(d)
    out, lse = varlen_attn_with_lse(qd, ent, True, hkv, scale)
    kd, vd = k.to(dev), v.to(dev)
    o2, l2 = ring_attn_with_lse(qd, kd, vd, scale, keys - new)
    cont, lc = varlen_attn_with_lse(qd, [make_entry(0, new, segment_contiguous(kd, vd), 0)],
                                    False, hkv, scale)
    torch.cuda.synchronize()
    o_ref, l_ref = orc.attn_with_lse(q, k, v, scale, keys - new)
    for o, l in ((out, lse), (o2, l2)):
        assert max_err(o, o_ref) <= OUT_TOL[torch.bfloat16]
        assert max_err(l, l_ref) <= LSE_TOL
    o_ref, l_ref = orc.attn_with_lse(q, k, v, scale, None)
    assert max_err(cont, o_ref) <= OUT_TOL[torch.bfloat16] and max_err(lc, l_ref) <= LSE_TOL


def test_split_under_capture_and_streams(dev):
    """A planned split replayed from a graph, in place over its accumulator,
    and on a side stream: every run equals the eager one."""
    h, hkv, d, tq, tk = 28, 4, 128, 64, 8192
    q, k, v = (t.to(dev) for t in _qkv(9, tq, tk, h, hkv, d, torch.bfloat16))
    acc_o, acc_l = ring_attn_with_lse(q, k[:300], v[:300], scale_for(d), None)

    def step(o, l):
        return ring_attn_merged(q, k, v, scale_for(d), tk - tq, o, l, output=o, output_lse=l)

    eo, el = acc_o.clone(), acc_l.clone()
    step(eo, el)
    go, gl = acc_o.clone(), acc_l.clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step(go, gl)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    assert torch.equal(go, eo) and torch.equal(gl, el)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step(go, gl)
    for _ in range(3):
        go.copy_(acc_o), gl.copy_(acc_l)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(go, eo) and torch.equal(gl, el)
        ring_attn_with_lse(q, k, v, scale_for(d), 0)


def test_no_room_for_the_partials(dev, monkeypatch):
    """Without memory for the workspace a launch that would be cut runs whole."""
    h, hkv, d, tq, tk = 14, 2, 64, 40, 9000
    q, k, v = _qkv(17, tq, tk, h, hkv, d, torch.bfloat16)
    asked = []
    monkeypatch.setattr(_lib, "scratch", lambda n, device: asked.append(n))
    o_ref, l_ref = orc.attn_with_lse(q, k, v, scale_for(d), tk - tq)
    qd, kd, vd = q.to(dev), k.to(dev), v.to(dev)
    for o, l in (ring_attn_with_lse(qd, kd, vd, scale_for(d), tk - tq),
                 varlen_attn_with_lse(qd, [make_entry(0, tq, segment_contiguous(kd, vd), tk - tq)],
                                      True, hkv, scale_for(d))):
        torch.cuda.synchronize()
        assert max_err(o, o_ref) <= OUT_TOL[torch.bfloat16] and max_err(l, l_ref) <= LSE_TOL
    assert len(asked) == 2 and all(n > 0 for n in asked)
