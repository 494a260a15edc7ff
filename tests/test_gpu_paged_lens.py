"""What the unplanned decode reads and when: the lengths once, in the split
kernel; the merge goes by the slots that kernel wrote, one pair for every
sequence.  In the backend these are the lengths that the host saw, and a layer
queued before that writes nothing unless the batch is a decode batch."""

import ctypes
import types

import pytest
import torch

from hcp_vllm_plugin_amd import _lib
from hcp_vllm_plugin_amd import ring_backend as rb
from hcp_vllm_plugin_amd.varlen import PagedCache, PagedDecode
from tests._util import OUT_TOL, max_err, scale_for
from tests.test_gpu_backend import _clean  # noqa: F401
from tests.test_gpu_decode_paged import _batch, _meta, _reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h,hkv,d", [(28, 4, 128), (6, 3, 64), (36, 2, 256)])
@pytest.mark.parametrize("lens", [[0], [0, 0, 900, 0, 33, 0], [700, 0, 0, 2000]])
def test_every_sequence_has_its_slots(dev, h, hkv, d, lens):
    n = len(lens)
    q, cache, bt = _batch(3, lens, h, hkv, d, torch.bfloat16, "v031", 16)
    pc, qd, btd = PagedCache.from_tensor(cache.to(dev)), q.to(dev), bt.to(dev)
    sl, out = torch.tensor(lens, dtype=torch.int32, device=dev), torch.full_like(qd, 7.0)
    a = PagedDecode(pc, btd, sl, h, None)._args
    ws = torch.full((a.workspace_bytes // 4,), 1 << 30, dtype=torch.int32, device=dev)
    a.q, a.q_stride_tok, a.q_stride_head = qd.data_ptr(), qd.stride(0), qd.stride(1)
    a.out, a.o_stride_tok, a.o_stride_head = out.data_ptr(), out.stride(0), out.stride(1)
    a.kv.k_addr, a.kv.v_addr, a.workspace = pc.k_addr, pc.v_addr, ws.data_ptr()
    a.scale, a.dtype = scale_for(d), _lib.dtype_code(qd.dtype)
    _lib.check(_lib.lib().hcp_decode_paged(ctypes.addressof(a), _lib.stream_ptr(dev)), "paged")
    torch.cuda.synchronize()
    slots = ws[-2 * n:].view(n, 2).tolist()
    end = 0  # slots lie in the order of the sequences
    for r, (first, last) in enumerate(slots):
        if lens[r] == 0:
            assert (first, last) == (0, -1) and torch.count_nonzero(out[r]) == 0
        else:
            assert end <= first <= last, slots
            end = last + 1


H, HKV, D = 28, 4, 128
LAYER = types.SimpleNamespace(layer_name="model.layers.0.self_attn.attn")


@pytest.mark.parametrize("qsl", [[0, 1, 2, 3], [0, 64, 65, 66]])
def test_lengths_refilled_for_the_next_step(dev, monkeypatch, qsl):
    """A layer waiting in its queue while another stream refills the lengths:
    it attends to the keys of its own step (the plain decode batch, and the
    single-token rows of a mixed one)."""
    monkeypatch.setattr(rb.HcpRingAttentionImpl, "_decode_rows_apart", lambda self, *a: True)
    lens = [900, 17, 2500]
    _, cache, bt = _batch(1, lens, H, HKV, D, torch.bfloat16, "v031", 16)
    meta = _meta(dev, qsl, lens, bt)
    gen = torch.Generator().manual_seed(2)
    q = torch.randn(qsl[-1], H, D, generator=gen).to(torch.bfloat16)
    qd, cached = q.to(dev), cache.to(dev)
    impl = rb.HcpRingAttentionImpl(H, D, scale_for(D), HKV)
    first, out = torch.empty_like(qd), torch.empty_like(qd)
    impl.forward(LAYER, qd, None, None, cached, meta, first)
    a = torch.randn(8192, 8192, device=dev)
    torch.cuda.synchronize()
    for _ in range(8):  # several milliseconds for the second layer to wait
        a = (a @ a).clamp_(-1, 1)
    impl.forward(LAYER, qd, None, None, cached, meta, out)
    side = torch.cuda.Stream(dev)
    with torch.cuda.stream(side):
        meta.seq_lens.fill_(1)
    side.synchronize()
    torch.cuda.synchronize()
    assert torch.equal(out, first)
    rows = [qsl[r + 1] - 1 for r in range(3)][-3 if qsl[1] == 1 else -2:]
    ref = _reference(q[rows], cache, bt[-len(rows):], lens[-len(rows):], "v031", scale_for(D), 0)
    assert max_err(out[rows], ref) <= OUT_TOL[torch.bfloat16]


def test_queued_ahead_writes_only_a_decode_batch(dev):
    """As many tokens as requests: rows that belong to no request, and the
    output of a refused batch, stay as they were."""
    lens = [900, 17, 30]
    q, cache, bt = _batch(4, lens, H, HKV, D, torch.bfloat16, "v031", 16)
    qd, cached = q.to(dev), cache.to(dev)
    impl = rb.HcpRingAttentionImpl(H, D, scale_for(D), HKV)
    out = torch.full_like(qd, 7.0)
    meta = _meta(dev, [0, 2, 2, 2], lens, bt)
    meta.num_actual_tokens = 3
    impl.forward(LAYER, qd, None, None, cached, meta, out)
    torch.cuda.synchronize()
    assert (out[2] == 7).all() and not (out[:2] == 7).all()
    out.fill_(7.0)
    for bad in ([900, 17, bt.shape[1] * 16 + 1], [900, -1, 30]):
        with pytest.raises(ValueError):
            impl.forward(LAYER, qd, None, None, cached, _meta(dev, [0, 1, 2, 3], bad, bt), out)
        torch.cuda.synchronize()
        assert (out == 7).all()


def test_a_step_that_failed_leaves_no_lengths_behind(dev):
    """A step refused while its first layer was being queued has written its
    lengths; the step before it, still the caller's, runs on its own."""
    lens, other = [900, 17, 2500], [5, 3, 7]
    q, cache, bt = _batch(1, lens, H, HKV, D, torch.bfloat16, "v031", 16)
    qd, cached = q.to(dev), cache.to(dev)
    impl = rb.HcpRingAttentionImpl(H, D, scale_for(D), HKV)
    meta = _meta(dev, [0, 1, 2, 3], lens, bt)
    first, second = torch.empty_like(qd), torch.empty_like(qd)
    impl.forward(LAYER, qd, None, None, cached, meta, first)
    odd = torch.zeros(cached.numel() + 1, dtype=qd.dtype, device=dev)[1:].view(cached.shape)
    with pytest.raises(ValueError, match="16-byte aligned"):
        impl.forward(LAYER, qd, None, None, odd, _meta(dev, [0, 1, 2, 3], other, bt), second)
    impl.forward(LAYER, qd, None, None, cached, meta, second)
    torch.cuda.synchronize()
    assert torch.equal(first, second)
    ref = _reference(q, cache, bt, lens, "v031", scale_for(D), 0)
    assert max_err(second, ref) <= OUT_TOL[torch.bfloat16]
