"""Mixed batches whose single-token rows run in the decode launch, against the
oracle: rows before, between and after the prefill chunks, with staged and
split peers, windows, prefixes past a row's position, and no prefill at all."""

import pytest
import torch

from hcp_vllm_plugin_amd import ring_backend as rb
from tests.test_gpu_backend import _clean, _run  # noqa: F401

pytestmark = pytest.mark.gpu

REQS = [(1, 700), (300, 900), (1, 1), (1, 2050), (17, 517), (0, 64), (1, 40)]
CHUNKS = [[64, 128], [64], None, [1024], None, None, [48]]


@pytest.mark.parametrize("layout", ["v031", "v023"])
@pytest.mark.parametrize("window", [None, 100])
@pytest.mark.parametrize("peer", ["none", "staged", "split"])
def test_mixed_rows_apart(dev, monkeypatch, layout, window, peer):
    monkeypatch.setattr(rb.HcpRingAttentionImpl, "_decode_rows_apart", lambda self, *a: True)
    _run(dev, layout, REQS, staged_chunks=CHUNKS if peer == "staged" else None,
         split=650 if peer == "split" else 0, monkeypatch=monkeypatch, window=window)
    assert rb.IMPL_STATS["decode_hip"] == 1 and rb.IMPL_STATS["attn_hip"] >= 1


def test_rows_without_any_prefill(dev, monkeypatch):
    """An empty request among single-token rows: not the plain decode batch
    (row r is not request r), every row in the decode launch."""
    monkeypatch.setattr(rb.HcpRingAttentionImpl, "_decode_rows_apart", lambda self, *a: True)
    _run(dev, "v031", [(1, 333), (0, 64), (1, 900)], dtype=torch.float16)
    assert rb.IMPL_STATS["decode_hip"] == 1 and rb.IMPL_STATS["attn_hip"] == 0


def test_long_rows_leave_the_prefill_launch(dev):
    """The rule itself: 28 heads, 24k keys in single-token rows."""
    _run(dev, "v031", [(64, 200), (1, 9000), (1, 15500)])
    assert rb.IMPL_STATS["decode_hip"] == 1 and rb.IMPL_STATS["attn_hip"] == 1
