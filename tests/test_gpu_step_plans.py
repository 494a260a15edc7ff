"""Plans that the layers of a step share, against the oracle: on other layers'
caches, on another stream than the step began on, over staged peers whose
chunks differ per layer; and the unplanned decode over block tables with padded
rows and other block sizes."""

import types

import pytest
import torch

from hcp_vllm_plugin_amd import ring_backend as rb
from hcp_vllm_plugin_amd.varlen import PagedCache, PagedDecode
from oracle import ring_oracle as orc
from tests._util import OUT_TOL, max_err, randn, scale_for
from tests.test_gpu_backend import _clean  # noqa: F401
from tests.test_gpu_decode_paged import _batch, _gather, _meta, _reference

pytestmark = pytest.mark.gpu

H, HKV, D = 28, 4, 128
REQS = {"prefill": [(200, 900), (64, 64), (1, 30)],
        "mixed": [(64, 300), (1, 9000), (1, 15500), (17, 200)],
        "decode": [(1, 900), (1, 17), (1, 2500)]}


def _layer(seed, lens, rows, layout, bs):
    """A layer's q and cache; the block table is the same for every seed."""
    _, cache, bt = _batch(11, lens, H, HKV, D, torch.bfloat16, layout, bs)
    gen = torch.Generator().manual_seed(seed)
    cache = randn(gen, tuple(cache.shape), torch.bfloat16)
    return randn(gen, (rows, H, D), torch.bfloat16), cache, bt


def _expect(q, cache, bt, reqs, layout, peers=None):
    ref, at = torch.zeros(q.shape), 0
    for r, (t, n) in enumerate(reqs):
        k, v = _gather(cache.float(), layout, bt[r], n)
        if peers and peers[r] is not None:
            p = peers[r][0].shape[0]
            k, v = torch.cat([peers[r][0].float(), k[p:]]), torch.cat([peers[r][1].float(), v[p:]])
        ref[at:at + t] = orc.attn_with_lse(q[at:at + t].float(), k, v, scale_for(D), n - t)[0]
        at += t
    return ref


def _ok(out, ref):
    return max_err(out, ref) <= OUT_TOL[torch.bfloat16] * max(1.0, ref.abs().max().item() / 4)


@pytest.mark.parametrize("layout", ["v031", "v023"])
@pytest.mark.parametrize("kind", list(REQS))
@pytest.mark.parametrize("bs", [8, 16, 32])
def test_three_layers_on_two_streams(dev, layout, kind, bs):
    """Layer 0 plans; layer 1 has another cache; layer 2 and a second pass of
    layer 0 run on another stream (which waits for the first), with the next
    step queued before any of it is waited for."""
    reqs = REQS[kind]
    qsl = [0]
    for t, _ in reqs:
        qsl.append(qsl[-1] + t)
    lens = [n for _, n in reqs]
    impl = rb.HcpRingAttentionImpl(H, D, scale_for(D), HKV)
    layers = [_layer(20 + i, lens, qsl[-1], layout, bs) for i in range(3)]
    on = [(q.to(dev), c.to(dev), torch.full(q.shape, 7.0, dtype=q.dtype, device=dev))
          for q, c, _ in layers]
    bt = layers[0][2]
    metas = [_meta(dev, qsl, lens, bt) for _ in range(2)]
    again = torch.full_like(on[0][2], 7.0)
    side = torch.cuda.Stream(dev)
    torch.cuda.synchronize()

    def run(i, meta, out=None):
        q, c, o = on[i]
        lay = types.SimpleNamespace(layer_name="model.layers.%d.self_attn.attn" % i)
        impl.forward(lay, q, None, None, c, meta, o if out is None else out)

    run(0, metas[0])
    run(1, metas[0])
    side.wait_stream(torch.cuda.current_stream(dev))
    with torch.cuda.stream(side):
        run(2, metas[0])
        run(0, metas[0], again)
    metas[0].seq_lens.fill_(1)  # the first step is queued; its lengths are its own
    second = torch.full_like(again, 7.0)
    run(0, metas[1], second)
    torch.cuda.synchronize()
    for i, (q, c, b) in enumerate(layers):
        assert _ok(on[i][2], _expect(q, c, b, reqs, layout)), i
    assert torch.equal(again, on[0][2]) and torch.equal(second, on[0][2])


@pytest.mark.parametrize("layout", ["v031", "v023"])
def test_staged_prefill_layers(dev, layout):
    """A local plan shared by layers with chunks of the same length, and one of
    its own for a layer whose chunk is shorter."""
    reqs, lens = [(100, 400), (1, 200), (30, 90)], [400, 200, 90]
    qsl = [0, 100, 101, 131]
    impl = rb.HcpRingAttentionImpl(H, D, scale_for(D), HKV)
    layers = [_layer(40 + i, lens, 131, layout, 16) for i in range(3)]
    bt = layers[0][2]
    bt[:, 0] = torch.arange(3, dtype=torch.int32)  # names of the requests
    meta = _meta(dev, qsl, lens, bt)
    rb.map_request_peer(0, ["a"])
    rb.map_request_peer(1, ["b"])
    gen = torch.Generator().manual_seed(9)
    for i, (q, c, _) in enumerate(layers):
        name = "model.layers.%d.self_attn.attn" % i
        peers = []
        for ck, n in (("a", 304 if i < 2 else 160), ("b", 64)):
            kv = randn(gen, (n, HKV, D), q.dtype), randn(gen, (n, HKV, D), q.dtype)
            rb.stage_peer_kv(ck, name, kv[0].to(dev), kv[1].to(dev))
            peers.append(kv)
        out = torch.full(q.shape, 7.0, dtype=q.dtype, device=dev)
        impl.forward(types.SimpleNamespace(layer_name=name), q.to(dev), None, None, c.to(dev),
                     meta, out)
        torch.cuda.synchronize()
        ref = _expect(q, c, bt, reqs, layout, peers + [None])
        # rows inside the prefix see local keys alone (n_a of them)
        n_a = max(0, min(100, peers[0][0].shape[0] - 300))
        if n_a:
            k, v = _gather(c.float(), layout, bt[0], 400)
            ref[:n_a] = orc.attn_with_lse(q[:n_a].float(), k, v, scale_for(D), 300)[0]
        assert _ok(out, ref), i
    assert sum(1 for k in rb._STEP["fast"] if k[0] == "local") == 2


@pytest.mark.parametrize("bs", [1, 4, 16, 64, 256])
@pytest.mark.parametrize("layout,pad,wide,window", [("v031", 0, False, 0), ("v023", 5, True, 70),
                                                    ("v031", 3, False, 300)])
def test_unplanned_decode_tables(dev, bs, layout, pad, wide, window):
    """Rows of the block table ``pad`` elements apart, which name blocks past
    the cache; any block size."""
    lens = [500, 0, 33, 1700, 1]
    q, cache, bt = _batch(bs + pad, lens, H, HKV, D, torch.float16, layout, bs)
    held = torch.full((len(lens), bt.shape[1] + pad), 1 << 30, dtype=torch.int32)
    held[:, :bt.shape[1]] = bt
    table = held.to(dev)[:, :bt.shape[1]]
    assert table.stride(0) == bt.shape[1] + pad
    sl = torch.tensor(lens, dtype=torch.int64 if wide else torch.int32, device=dev)
    pc, qd = PagedCache.from_tensor(cache.to(dev)), q.to(dev)
    assert PagedDecode.takes(table, sl, bs)
    out = torch.full_like(qd, 7.0)
    PagedDecode(pc, table, sl, H, window or None).run(qd, out, pc, scale_for(D))
    torch.cuda.synchronize()
    ref = _reference(q, cache, bt, lens, layout, scale_for(D), window)
    assert max_err(out, ref) <= OUT_TOL[torch.float16] * max(1.0, ref.abs().max().item() / 4)
