"""What the KV-split planners keep to, and the memory a cut launch takes: one
source for the limits, a bounded workspace, reserved by the profiling run and
not asked for in every layer when there is no room.  On the CPU."""

import ctypes
import os
import re
import types

import pytest
import torch

from hcp_vllm_plugin_amd import _lib
from hcp_vllm_plugin_amd import ring_backend as rb

HEADER = os.path.join(os.path.dirname(_lib.__file__), "..", "include", "hcp_mi355x.h")


def _plan(tq, tk, h, hkv, d, off=None, window=0):
    whole, nbytes = ctypes.c_int32(0), ctypes.c_size_t(0)
    pt = _lib.lib().hcp_plan_fwd_split(tq, tk, h, hkv, d, int(off is not None), off or 0, window,
                                       ctypes.addressof(whole), ctypes.addressof(nbytes))
    assert pt >= 0
    return pt, nbytes.value


@pytest.mark.parametrize("h,hkv,d,tq,tk,off", [
    (28, 4, 128, 941, 175090, None), (64, 8, 128, 136, 199547, 199411),
    (16, 8, 256, 924, 164181, None), (14, 2, 64, 6924, 4182, -2742),
    # blocks of very unequal length: as many slots each as the longest has pieces
    (8, 8, 128, 16051, 1974, -14077), (1, 1, 128, 125171, 15344, -109827),
    (4, 1, 256, 28509, 86509, -21566), (8, 2, 128, 4000, 9000, 100),
])
def test_workspace_stays_within_the_limit(h, hkv, d, tq, tk, off):
    lim = _lib.split_limits(d)
    assert lim.max_workspace == lim.max_pieces * 128 * ((64 if d == 64 else d) + 1) * 4
    assert _plan(tq, tk, h, hkv, d, off)[1] <= lim.max_workspace


@pytest.mark.parametrize("h,hkv,d", [(28, 4, 128), (14, 2, 64), (16, 8, 256), (1, 1, 128)])
def test_what_is_not_asked_about_is_never_cut(h, hkv, d):
    lim = _lib.split_limits(d)
    for tq in (1, 33, 128, 300):
        assert _plan(tq, lim.min_keys - 1, h, hkv, d)[0] == 0
        assert _plan(tq, lim.min_keys - 1, h, hkv, d, lim.min_keys - 1 - tq)[0] == 0
    blocks = lim.max_units // h + 1
    for tk in (5000, 100000):
        assert _plan(blocks * 128, tk, h, hkv, d)[0] == 0
    # ... and these are
    assert _plan(512, 32768, 28, 4, 128, 32256)[0] > 0
    assert _plan(16, 8192, h, hkv, d)[0] > 0


def test_limits_of_other_head_sizes():
    assert _lib.split_limits(80) == _lib.split_limits(128)
    assert _lib.split_limits(512).max_units == 0  # the launch refuses it
    with open(HEADER) as f:
        text = f.read()
    assert int(re.search(r"HCP_DECODE_PAGED_MAX_SEQS (\d+)", text)[1]) == _lib.DECODE_PAGED_MAX_SEQS


def test_no_room_is_remembered_for_a_while(monkeypatch):
    dev, asked, now = torch.device("cpu"), [], [100.0]
    room = [1000]

    def empty(n, **kw):
        asked.append(n)
        if n > room[0]:
            raise torch.OutOfMemoryError("no room")
        return "memory"

    monkeypatch.setattr(_lib.torch, "empty", empty)
    monkeypatch.setattr(_lib.time, "monotonic", lambda: now[0])
    monkeypatch.setattr(_lib, "_no_room", {})
    assert _lib.scratch(2000, dev) is None
    for n in (2000, 3000, 2500):  # the layers that follow
        assert _lib.scratch(n, dev) is None
    assert asked == [2000]
    assert _lib.scratch(900, dev) == "memory"  # less than that is another question
    assert _lib.scratch(2000, dev) is None and asked == [2000, 900]
    room[0] = 5000
    assert _lib.scratch(2000, dev) is None
    now[0] += 1.5
    assert _lib.scratch(2000, dev) == "memory" and _lib.scratch(3000, dev) == "memory"


def test_profiling_run_has_the_partials(monkeypatch):
    asked = []
    monkeypatch.setattr(_lib, "scratch", lambda n, device: asked.append((n, device)))
    capturing = [False]
    monkeypatch.setattr(rb, "_capturing", lambda: capturing[0])
    out = types.SimpleNamespace(is_cuda=True, device="gpu", fill_=lambda v: ("filled", v))
    impl = rb.HcpRingAttentionImpl(28, 80, 0.1, 4)
    assert impl.forward(None, None, None, None, None, None, out) == ("filled", 0)
    assert asked == [(_lib.split_limits(80).max_workspace, "gpu")]
    capturing[0] = True  # not into a graph's pool
    assert impl.forward(None, None, None, None, None, None, out) == ("filled", 0)
    cpu = torch.ones(2, 2)
    assert impl.forward(None, None, None, None, None, None, cpu).sum() == 0 and len(asked) == 1


# (query rows, keys) of a launch of one request: pieces, at least
@pytest.mark.parametrize("heads,causal,window,new,keys,least", [
    ((28, 4, 128), 1, 0, 512, 32768, 4 * 4), ((28, 4, 128), 0, 0, 512, 32768, 4 * 4),
    ((14, 2, 64), 1, 0, 512, 32768, 4 * 4), ((16, 8, 256), 1, 0, 512, 32768, 4 * 2),
    ((12, 3, 128), 0, 0, 16, 4099, 2), ((28, 4, 128), 1, 0, 16, 4099, 2),
    ((28, 4, 128), 1, 700, 16, 4099, 1),  # the window's 12 tiles: whole
])
def test_varlen_launches_that_are_cut(heads, causal, window, new, keys, least):
    from tests.test_split_plan import _entries, _plan as plan_varlen

    pieces, units, slots, _, nbytes = plan_varlen(_entries([(0, new, keys)], causal), causal,
                                                  window, heads)
    if least == 1:
        assert len(pieces) == 0 and nbytes == 0
        return
    assert len(pieces) >= least and len(units) >= 1 and slots >= 2
    assert 0 < nbytes <= _lib.split_limits(heads[2]).max_workspace
