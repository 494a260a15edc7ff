"""NaN and infinite inputs: a row comes out as the launch that is not cut (or
the batch that is not taken apart) gives it, on whatever kernels it runs."""

import types

import pytest
import torch

from hcp_vllm_plugin_amd import ring_backend as rb
from hcp_vllm_plugin_amd.varlen import PagedCache, PagedDecode, decode_attn, segment_contiguous
from hcp_vllm_plugin_amd import ring_attn_merged, ring_attn_with_lse
from tests._util import randn, scale_for
from tests.test_gpu_backend import _clean  # noqa: F401
from tests.test_gpu_decode_paged import _batch, _meta
from tests.test_gpu_split import _qkv, _split

pytestmark = pytest.mark.gpu

NAN, INF = float("nan"), float("inf")


def _same(got, want, tol, strict=True):
    """NaN and infinities in the same places, the rest within ``tol``.  Not
    ``strict``: infinite or NaN alike -- an infinite V meets a P that is 0 in 16
    bits (and gives NaN) relative to one maximum and not to another."""
    got, want = got.float(), want.float()
    assert torch.equal(torch.isfinite(got), torch.isfinite(want))
    if strict:
        assert torch.equal(torch.isnan(got), torch.isnan(want))
        assert torch.equal(got == INF, want == INF) and torch.equal(got == -INF, want == -INF)
    ok = torch.isfinite(want)
    assert not ok.any() or (got[ok] - want[ok]).abs().max().item() <= tol


def _poison(q, k, v, what):
    """``what`` at one query row, at keys of one or several pieces, or in V."""
    if what == "q":
        q[5, 1, 3], q[40, 0, 0] = NAN, INF
    elif what == "k":
        k[700, :, 1] = NAN
    elif what == "k all":
        k[:, 0, 1] = NAN
    elif what == "k inf":
        k[3, :, 2] = INF
    else:
        v[700, :, 4], v[100, :, 5] = NAN, INF
    return q, k, v


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("h,hkv,d", [(8, 2, 128), (4, 2, 64), (4, 4, 256)])
@pytest.mark.parametrize("what", ["q", "k", "k all", "k inf", "v"])
@pytest.mark.parametrize("off,window", [(None, 0), (872, 0), (872, 400)])
def test_cut_prefill_rows(dev, dtype, h, hkv, d, what, off, window):
    tq, tk = 150, 1000
    q, k, v = (x.to(dev) for x in _poison(*_qkv(d, tq, tk, h, hkv, d, dtype), what))
    scale = scale_for(d)
    whole, whole_l = _split(q, k, v, scale, off, window, 100, 0)  # one piece: nothing is cut
    acc_o = randn(torch.Generator().manual_seed(1), (tq, h, d), dtype).to(dev)
    acc_l = torch.full((h, tq), 1.0, device=dev)
    acc_l[:, 3:9] = -INF
    want, want_l = _split(q, k, v, scale, off, window, 100, 0, (acc_o, acc_l))
    # P and the output round to the dtype, the partials to f32
    tol = 2.0 ** (-8 if dtype == torch.bfloat16 else -11) * 4 * max(
        1.0, whole.float().nan_to_num(0, 0, 0).abs().max().item())
    for piece in (1, 4):
        out, lse = _split(q, k, v, scale, off, window, piece, 0)
        _same(out, whole, tol, what != "v")
        _same(lse, whole_l, 1e-3)
        out, lse = _split(q, k, v, scale, off, window, piece, 0, (acc_o, acc_l))
        _same(out, want, tol, what != "v")
        _same(lse, want_l, 1e-3)


def test_planned_cut_and_whole_agree(dev):
    """The entry points, where the planner cuts: a NaN query row is NaN."""
    q, k, v = _qkv(1, 16, 8192, 14, 2, 64, torch.bfloat16)
    q[7] = NAN
    qd, kd, vd = q.to(dev), k.to(dev), v.to(dev)
    out, lse = ring_attn_with_lse(qd, kd, vd, scale_for(64), None)
    assert torch.isnan(out[7]).all() and (lse[:, 7] == -INF).all()
    rest = [i for i in range(16) if i != 7]
    assert torch.isfinite(out[rest]).all() and torch.isfinite(lse[:, rest]).all()
    merged = ring_attn_merged(qd, kd, vd, scale_for(64), None, torch.ones_like(out),
                              torch.zeros_like(lse))
    assert (merged[7] == 1).all()  # a side without weight, as in the merge after a whole pass


@pytest.mark.parametrize("lens", [[200, 9000, 40, 5000], [9000, 200, 40, 700]])
@pytest.mark.parametrize("peers", ["none", "staging of others", "staged"])
def test_single_token_rows_of_a_mixed_batch(dev, monkeypatch, lens, peers):
    """Rows with NaN in q, or in one key, as the prefill launch gives them,
    unplanned and planned; next to a staged peer, which the prefill launches
    merge with, a row of NaN scores has no weight."""
    h, hkv, d = 8, 2, 128
    tq = [1, 64, 1, 1] if lens[0] == 200 else [64, 1, 1, 1]
    qsl = [0]
    for t in tq:
        qsl.append(qsl[-1] + t)
    _, cache, bt = _batch(7, lens, h, hkv, d, torch.bfloat16, "v031", 16)
    if peers != "staged":  # one key of the third request, in a block of its own
        cache[bt[2, 1], :, 3, 5] = NAN
    gen = torch.Generator().manual_seed(2)
    q = randn(gen, (qsl[-1], h, d), torch.bfloat16)
    q[qsl[-1] - 1] = NAN
    impl = rb.HcpRingAttentionImpl(h, d, scale_for(d), hkv)
    layer = types.SimpleNamespace(layer_name="model.layers.0.self_attn.attn")
    bt[:, 0] = torch.arange(4, dtype=torch.int32)  # the requests' names, still blocks of the cache
    if peers == "staging of others":
        rb.stage_peer_kv("c", "another.layer", torch.zeros(16, hkv, d, dtype=q.dtype, device=dev),
                         torch.zeros(16, hkv, d, dtype=q.dtype, device=dev))
        rb.map_request_peer(2, ["c"])
    elif peers == "staged":
        for r in (1, 2):
            rb.stage_peer_kv("c%d" % r, layer.layer_name,
                             randn(gen, (32, hkv, d), q.dtype).to(dev),
                             randn(gen, (32, hkv, d), q.dtype).to(dev))
            rb.map_request_peer(r, ["c%d" % r])
    got = []
    for apart in (False, True):
        monkeypatch.setattr(rb.HcpRingAttentionImpl, "_decode_rows_apart",
                            lambda self, *a, apart=apart: apart)
        out = torch.full((qsl[-1], h, d), 7.0, dtype=q.dtype, device=dev)
        impl.forward(layer, q.to(dev), None, None, cache.to(dev), _meta(dev, qsl, lens, bt), out)
        torch.cuda.synchronize()
        got.append(out)
    assert rb.IMPL_STATS["decode_hip"] == 1
    bad = got[0].float()
    if peers == "staged":
        assert torch.isfinite(bad).all() and (bad[-1] == 0).all()
    else:
        assert torch.isnan(bad[-1]).all() and torch.isnan(bad[qsl[2]]).all()
    _same(got[1], got[0], 2 * 1.5e-2)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("h,hkv,d", [(8, 2, 128), (4, 2, 64), (4, 4, 256)])
def test_decode_with_infinite_values(dev, dtype, h, hkv, d):
    """An infinite V element makes its output column infinite, with its sign,
    whatever its key's weight rounds to (the largest weight of the row, 1,
    among them); the other columns stay what they are."""
    n = 1500
    gen = torch.Generator().manual_seed(d)
    q = randn(gen, (2, h, d), dtype) * 0.2
    k, v = randn(gen, (n, hkv, d), dtype), randn(gen, (n, hkv, d), dtype)
    kd = k.float().reshape(n, hkv, d).repeat_interleave(h // hkv, 1)
    sc = torch.einsum("thd,nhd->thn", q.float(), kd) * scale_for(d)
    top = sc.argmax(-1)[0]  # the first row's heaviest key of each head
    keys = torch.unique(torch.cat([top, torch.tensor([0, 31, 32, 700, n - 2])]))
    inf = v.clone()
    for i, key in enumerate(keys.tolist()):
        inf[key, :, i] = INF if i % 2 else -INF
    col = torch.arange(len(keys))
    pc_cache = torch.zeros(100, hkv, 16, 2 * d, dtype=dtype)
    pc_cache[torch.arange(n) // 16, :, torch.arange(n) % 16] = torch.cat([k, inf], -1)
    cache = pc_cache.to(dev)
    bt = torch.arange(100, dtype=torch.int32, device=dev).repeat(2, 1)
    lens = torch.tensor([n, n], dtype=torch.int32, device=dev)
    qd, kdev, vdev, idev = q.to(dev), k.to(dev), v.to(dev), inf.to(dev)
    want = decode_attn(qd, [[segment_contiguous(kdev, vdev)]] * 2, hkv, scale_for(d))
    flat = decode_attn(qd, [[segment_contiguous(kdev, idev)]] * 2, hkv, scale_for(d))
    paged = torch.empty_like(flat)
    pc = PagedCache.from_tensor(cache)
    PagedDecode(pc, bt, lens, h, None).run(qd, paged, pc, scale_for(d))
    torch.cuda.synchronize()
    ref = torch.where(col % 2 == 1, INF, -INF).to(dev)
    tol = 2.0 ** (-8 if dtype == torch.bfloat16 else -11) * 4
    for out in (flat, paged):
        hit = out[..., :len(keys)].float()
        assert (hit == ref).all(), [(keys[c].item(), hit[..., c].tolist()) for c in col if not (hit[..., c] == ref[c]).all()]
        assert (out[..., len(keys):].float() - want[..., len(keys):].float()).abs().max() <= tol
