"""What the unplanned decode reads and when: the lengths once, in the split
kernel; the merge goes by the slots that kernel wrote, one pair for every
sequence."""

import ctypes

import pytest
import torch

from hcp_vllm_plugin_amd import _lib
from hcp_vllm_plugin_amd.varlen import PagedCache, PagedDecode
from tests._util import scale_for
from tests.test_gpu_decode_paged import _batch

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
