"""The backend's host side of a step, on the CPU: metadata that does not fit
together is refused before anything is queued."""

import types

import numpy as np
import pytest
import torch

from hcp_vllm_plugin_amd import ring_backend as rb
from hcp_vllm_plugin_amd.varlen import PagedCache, PagedDecode, paged_entry_array


@pytest.fixture(autouse=True)
def _clean():
    rb.invalidate_step_cache()
    yield
    rb.invalidate_step_cache()


def _meta(qsl, lens, bt):
    return types.SimpleNamespace(
        num_actual_tokens=qsl[-1], query_start_loc=torch.tensor(qsl, dtype=torch.int32),
        seq_lens=torch.tensor(lens, dtype=torch.int32),
        block_table=torch.tensor(bt, dtype=torch.int32))


def _forward(meta):
    impl = rb.HcpRingAttentionImpl(4, 64, 0.125, 2)
    layer = types.SimpleNamespace(layer_name="model.layers.0.self_attn.attn")
    q = torch.zeros(meta.num_actual_tokens, 4, 64, dtype=torch.bfloat16)
    cache = torch.zeros(8, 2, 16, 128, dtype=torch.bfloat16)
    return impl.forward(layer, q, None, None, cache, meta, torch.zeros_like(q))


@pytest.mark.parametrize("qsl", [[0, 1, 2, 3], [0, 4, 5, 9]])
def test_block_table_without_a_row_for_a_request(qsl):
    with pytest.raises(ValueError, match="no row for a request"):
        _forward(_meta(qsl, [20, 20, 20], [[0, 1], [2, 3]]))


def test_block_table_rows_of_entries_and_unplanned_batches():
    pc = PagedCache.from_tensor(torch.zeros(8, 2, 16, 128, dtype=torch.bfloat16))
    bt = torch.zeros(2, 4, dtype=torch.int32)
    for rows, lens in (([0, 2], [5, 5]), ([-1, 0], [5, 5])):
        with pytest.raises(ValueError, match="no row for a request"):
            paged_entry_array(pc, bt, rows, rows, 1, 0, 0, np.asarray(lens))
    # a row that nothing is read through may lie past the table
    assert len(paged_entry_array(pc, bt, [0, 2], [0, 1], 1, 0, 0, np.asarray([5, 0]))) == 2
    with pytest.raises(ValueError, match="no row for a request"):
        PagedDecode(pc, bt, torch.ones(3, dtype=torch.int32), 4, None)

    def on_gpu(t):  # what `takes` looks at
        return types.SimpleNamespace(shape=t.shape, dtype=t.dtype, stride=t.stride, dim=t.dim,
                                     is_cuda=True)

    lens = on_gpu(torch.ones(2, dtype=torch.int32))
    assert PagedDecode.takes(on_gpu(bt), lens, 16)
    assert not PagedDecode.takes(on_gpu(bt[:1]), lens, 16)
    assert not PagedDecode.takes(on_gpu(bt[0]), lens, 16)


def test_another_threads_step_leaves_a_layers_plans_alone(monkeypatch):
    """While a layer plans, another thread's step replaces the newest one: the
    layer goes on with its own plans, which the other step does not get."""
    mine, other = _meta([0, 3, 8], [20, 30], [[0, 1], [2, 3]]), _meta([0, 2], [9], [[4, 5]])
    calls = []

    def planner(name):
        def plan(self, *a):
            calls.append(name)
            rb._host_metadata(other)
        return plan

    monkeypatch.setattr(rb._lib, "stream_ptr", lambda device: 0)
    monkeypatch.setattr(rb, "_capturing", lambda: False)
    monkeypatch.setattr(rb.HcpRingAttentionImpl, "_plan_rows", planner("rows"))
    monkeypatch.setattr(rb.HcpRingAttentionImpl, "_plan_chunks", planner("chunks"))
    _forward(mine)
    assert calls == ["rows", "chunks"]
    assert rb._host_metadata(other)[0][1] == [9] and not rb._STEP["fast"]


@pytest.mark.parametrize("heads,d,rows,window,each_layer,apart", [
    (28, 128, [16384] * 2, None, False, True),
    (28, 128, [16384] * 2, 128, False, False),   # the prefill launch reads the window alone
    (28, 128, [16384] * 64, 128, False, False),
    (28, 128, [16384] * 64, 4096, False, True),
    (28, 128, [4096] * 8, None, False, True),
    (14, 64, [4096] * 8, None, False, False),    # half the columns, half the heads
    (14, 64, [4096] * 32, None, False, True),
    (16, 256, [4096] * 8, None, False, True),
    (28, 128, [5120] * 32, None, True, False),   # a plan in every layer costs more
    (28, 128, [9216] * 32, None, True, False),
    (28, 128, [17408] * 32, None, True, True),
    (28, 128, [25600] * 2, None, True, False),
    (28, 128, [50176] * 2, None, True, True),
    (28, 128, [], None, False, False),
])
def test_rows_that_leave_the_prefill_launch(heads, d, rows, window, each_layer, apart):
    """Next to two prefill chunks of many keys, which do not count."""
    impl = rb.HcpRingAttentionImpl(heads, d, 0.125, 2, sliding_window=window)
    qsl, lens = [0, 300], [60000]
    for n in rows:
        qsl.append(qsl[-1] + 1)
        lens.append(n)
    qsl.append(qsl[-1] + 300)
    lens.append(60000)
    assert impl._decode_rows_apart(qsl, lens, *([True] if each_layer else [])) == apart


def test_whose_lengths_a_launch_reads(monkeypatch):
    """The step's own on the thread and stream that wrote them; anywhere else a
    copy of the host's, one for each stream; the caller's under capture."""
    import threading

    words = torch.zeros(4, dtype=torch.int64)
    step = rb._Step(None, None, ([0, 1, 2], [70, 80], [0, 1]), None, words[2:],
                    (threading.get_ident(), 5))
    given = torch.ones(2, dtype=torch.int32)
    capturing = [False]
    monkeypatch.setattr(rb, "_capturing", lambda: capturing[0])
    monkeypatch.setattr(rb, "_upload", lambda arrays, device: (
        torch.from_numpy(np.concatenate([a.view(np.uint8) for a in arrays])), [0]))
    assert step.lens_on(5, None, given) is step.lens
    other = step.lens_on(6, None, given)
    assert other.tolist() == [70, 80] and step.lens_on(6, None, given) is other
    seen = []
    t = threading.Thread(target=lambda: seen.append(step.lens_on(5, None, given)))
    t.start()
    t.join()
    assert seen[0].tolist() == [70, 80] and seen[0].data_ptr() != step.lens.data_ptr()
    capturing[0] = True
    assert step.lens_on(5, None, given) is given
    capturing[0] = False
    step.lens = None  # metadata that came another way: nothing runs unplanned
    assert step.lens_on(5, None, given) is None
