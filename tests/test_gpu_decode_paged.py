"""Decode over a paged cache without a plan (``PagedDecode`` /
``hcp_decode_paged``), against the oracle: shares that end inside, at and
between sequences, empty sequences, windows, either index type, head groups
over 16, up to the largest batch -- and the backend queueing it before it has
seen the metadata."""

import types

import pytest
import torch

from hcp_vllm_plugin_amd import ring_backend as rb
from hcp_vllm_plugin_amd.varlen import PagedCache, PagedDecode
from oracle import ring_oracle as orc
from tests._util import OUT_TOL, max_err, outlier_k, randn, scale_for
from tests.test_gpu_backend import _clean  # noqa: F401

pytestmark = pytest.mark.gpu


def _batch(seed, lens, h, hkv, d, dtype, layout, bs):
    gen = torch.Generator().manual_seed(seed)
    need = [-(-n // bs) for n in lens]
    nb = sum(need) + 2
    shape = (nb, hkv, bs, 2 * d) if layout == "v031" else (nb, 2, bs, hkv, d)
    cache = randn(gen, shape, torch.float32)
    if layout == "v031":
        cache[..., :d] = outlier_k(cache[..., :d], gen)
    cache = cache.to(dtype)
    perm = torch.randperm(nb, generator=gen).to(torch.int32)
    bt = torch.full((len(lens), max(need) + 2), nb + 7, dtype=torch.int32)
    at = 0
    for r, n in enumerate(need):
        bt[r, :n] = perm[at:at + n]
        at += n
    return randn(gen, (len(lens), h, d), dtype), cache, bt


def _reference(q, cache, bt, lens, layout, scale, window):
    ref = torch.zeros(q.shape, dtype=torch.float32)
    for r, n in enumerate(lens):
        if n == 0:
            continue
        k, v = _gather(cache.float(), layout, bt[r], n)
        ref[r] = orc.attn_with_lse(q[r:r + 1].float(), k, v, scale, n - 1, window or None)[0][0]
    return ref


def _gather(cache, layout, row, n):
    bs = cache.shape[2]
    ids = row[:-(-n // bs)].long()
    if layout == "v031":
        kv = cache[ids].permute(0, 2, 1, 3).reshape(-1, cache.shape[1], cache.shape[3])[:n]
        return kv.chunk(2, -1)
    return tuple(cache[ids, i].reshape(-1, *cache.shape[3:])[:n] for i in (0, 1))


LENS = [
    [1], [63], [2000], [33, 1, 64, 31, 32],
    [0, 500, 0, 0, 1700, 3, 0],             # sequences without keys, first and last too
    [5000, 40, 40, 40, 40, 40, 6000],       # shares that cross many short sequences
    [700] * 33,
    [(37 * i) % 190 + 1 for i in range(200)],
]


@pytest.mark.parametrize("h,hkv,d", [(28, 4, 128), (14, 2, 64), (4, 2, 256), (36, 2, 128), (6, 3, 80)])
@pytest.mark.parametrize("lens", LENS, ids=range(len(LENS)))
@pytest.mark.parametrize("layout,window,wide", [("v031", 0, False), ("v023", 300, True)])
def test_matches_oracle(dev, h, hkv, d, lens, layout, window, wide):
    dtype = torch.bfloat16 if wide else torch.float16
    q, cache, bt = _batch(sum(lens) + d, lens, h, hkv, d, dtype, layout, 16)
    pc = PagedCache.from_tensor(cache.to(dev))
    sl = torch.tensor(lens, dtype=torch.int64 if wide else torch.int32, device=dev)
    btd, qd = bt.to(dev), q.to(dev)
    assert PagedDecode.takes(btd, sl, 16)
    out = torch.full_like(qd, 7.0)
    dec = PagedDecode(pc, btd, sl, h, window)
    dec.run(qd, out, pc, scale_for(d))
    torch.cuda.synchronize()
    ref = _reference(q, cache, bt, lens, layout, scale_for(d), window)
    # a row of few keys is close to one N(0, 1) value row, where bf16 rounds by
    # up to 2^-7 above 2 and 2^-6 above 4
    tol = OUT_TOL[dtype] * max(1.0, ref.abs().max().item() / 4)
    assert max_err(out, ref) <= tol
    again = torch.empty_like(out)
    dec.run(qd, again, pc, scale_for(d))
    torch.cuda.synchronize()
    assert torch.equal(again, out)


@pytest.mark.parametrize("n", [1024, 1023])
def test_largest_batch(dev, n):
    h, hkv, d = 8, 4, 64
    lens = [(i * 7919) % 97 for i in range(n)]
    q, cache, bt = _batch(5, lens, h, hkv, d, torch.float16, "v031", 16)
    pc = PagedCache.from_tensor(cache.to(dev))
    sl, out = torch.tensor(lens, dtype=torch.int32, device=dev), torch.empty_like(q, device=dev)
    PagedDecode(pc, bt.to(dev), sl, h, None).run(q.to(dev), out, pc, scale_for(d))
    torch.cuda.synchronize()
    ref = _reference(q, cache, bt, lens, "v031", scale_for(d), 0)
    assert max_err(out, ref) <= OUT_TOL[torch.float16] * max(1.0, ref.abs().max().item() / 4)
    assert not PagedDecode.takes(torch.zeros(1025, 4, dtype=torch.int32, device=dev),
                                 torch.ones(1025, dtype=torch.int32, device=dev), 16)


def _meta(dev, qsl, lens, bt):
    return types.SimpleNamespace(
        num_actual_tokens=qsl[-1], block_table=bt.to(dev),
        query_start_loc=torch.tensor(qsl, dtype=torch.int32, device=dev),
        seq_lens=torch.tensor(lens, dtype=torch.int32, device=dev))


def test_backend_queues_ahead(dev):
    """Three layers of a decode step; a batch of as many tokens as requests
    that is no decode batch (2 + 0 tokens), which runs again as a prefill; a
    length past the block table, refused as before."""
    h, hkv, d = 28, 4, 128
    lens = [900, 17, 2500]
    impl = rb.HcpRingAttentionImpl(h, d, scale_for(d), hkv)
    layer = types.SimpleNamespace(layer_name="model.layers.0.self_attn.attn")
    q, cache, bt = _batch(1, lens, h, hkv, d, torch.bfloat16, "v031", 16)
    meta = _meta(dev, [0, 1, 2, 3], lens, bt)
    for i in range(3):
        q, cache, _ = _batch(1 + i, lens, h, hkv, d, torch.bfloat16, "v031", 16)
        out = torch.full((3, h, d), 7.0, dtype=q.dtype, device=dev)
        impl.forward(layer, q.to(dev), None, None, cache.to(dev), meta, out)
        torch.cuda.synchronize()
        ref = _reference(q, cache, bt, lens, "v031", scale_for(d), 0)
        assert max_err(out, ref) <= OUT_TOL[torch.bfloat16], i
    assert rb.IMPL_STATS["decode_hip"] == 3 and rb.IMPL_STATS["attn_hip"] == 0

    two = _meta(dev, [0, 2, 2], [900, 17], bt[:2])
    out = torch.full((2, h, d), 7.0, dtype=q.dtype, device=dev)
    impl.forward(layer, q[:2].to(dev), None, None, cache.to(dev), two, out)
    torch.cuda.synchronize()
    k, v = _gather(cache.float(), "v031", bt[0], 900)
    ref = orc.attn_with_lse(q[:2].float(), k, v, scale_for(d), 898)[0]
    assert max_err(out, ref) <= OUT_TOL[torch.bfloat16]
    assert rb.IMPL_STATS["decode_hip"] == 3 and rb.IMPL_STATS["attn_hip"] == 1

    long = _meta(dev, [0, 1], [bt.shape[1] * 16 + 1], bt[2:])
    with pytest.raises(ValueError, match="block-table"):
        impl.forward(layer, q[:1].to(dev), None, None, cache.to(dev), long, out[:1])
    torch.cuda.synchronize()
