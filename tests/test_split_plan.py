"""The KV-split planners on the CPU: every (query block, tile) of a batch is in
exactly one piece, slots are used once, and a launch that fills the machine is
left whole (``hcp_plan_varlen_split``, ``hcp_plan_fwd_split``)."""

import ctypes

import numpy as np
import pytest

from hcp_vllm_plugin_amd import _lib
from hcp_vllm_plugin_amd.varlen import ENTRY_DTYPE

CAP = 4096


def _entries(reqs, causal):
    a = np.zeros(len(reqs), dtype=ENTRY_DTYPE)
    for i, (qs, n, keys) in enumerate(reqs):
        a[i] = (qs, n, keys - n if causal else 0, 4096, 4096, 0, 512, 128, 0, 0, keys, 0, 0)
    return a


def _plan(a, causal, window, heads):
    L = _lib.lib()
    pieces, units = np.zeros((CAP, 4), np.int32), np.zeros((CAP, 4), np.int32)
    nu, ns, pt = (ctypes.c_int32(0) for _ in range(3))
    nb = ctypes.c_size_t(0)
    rc = L.hcp_plan_varlen_split(a.ctypes.data, len(a), causal, window, *heads,
                                 pieces.ctypes.data, CAP, units.ctypes.data,
                                 ctypes.addressof(nu), ctypes.addressof(ns),
                                 ctypes.addressof(pt), ctypes.addressof(nb))
    _lib.check(rc, "plan")
    return pieces[:rc], units[:nu.value], ns.value, pt.value, nb.value


def _tiles(e, qb, causal, window):
    lo, hi = 0, int(e["len"])
    if causal:
        first = int(e["causal_offset"]) + qb * 128
        hi = min(hi, first + 128)
        if window:
            lo = min(max(0, first - window + 1), int(e["len"]))
    return -(-max(0, hi - lo) // 64)


@pytest.mark.parametrize("causal,window", [(1, 0), (1, 700), (0, 0)])
@pytest.mark.parametrize("heads", [(28, 4, 128), (14, 2, 64), (16, 8, 256), (12, 3, 128)])
@pytest.mark.parametrize("reqs", [
    [(0, 512, 32768)], [(0, 16, 4099)], [(0, 300, 20001), (300, 1, 9000), (301, 129, 129)],
    [(0, 700, 6000), (700, 700, 6000)], [(0, 5, 0), (5, 64, 30000)],
])
def test_varlen_split_covers_every_tile_once(reqs, heads, causal, window):
    a = _entries(reqs, causal)
    pieces, units, slots, pt, nbytes = _plan(a, causal, window, heads)
    if not len(pieces):
        return
    cut = {(int(e), int(b)): (int(s0), int(np_)) for e, b, s0, np_ in units}
    got: dict = {}
    for e, b, i, slot in pieces.tolist():
        got.setdefault((e, b), []).append((i, slot))
    want = {(i, b) for i, (_, n, _) in enumerate(reqs) for b in range(-(-n // 128))}
    assert set(got) == want
    used = set()
    for (e, b), lst in got.items():
        nt = _tiles(a[e], b, causal, window)
        if (e, b) not in cut:
            assert lst == [(0, -1)]
            continue
        s0, np_ = cut[(e, b)]
        # the kernel cuts a block of nt tiles into ceil(nt / pt) pieces
        assert np_ == -(-nt // pt) and np_ > 1
        assert sorted(lst) == [(i, s0 + i) for i in range(np_)]
        used.update(s for _, s in lst)
    assert used == set(range(slots))
    dw = 64 if heads[2] <= 64 else 128 if heads[2] <= 128 else 256
    assert nbytes == slots * heads[0] * 128 * (dw + 1) * 4


def test_full_launches_stay_whole():
    L = _lib.lib()
    w, nb = ctypes.c_int32(7), ctypes.c_size_t(7)
    for args in [(8192, 8192, 28, 4, 128, 1, 0, 0), (256, 256, 28, 4, 128, 1, 0, 0),
                 (8192, 8192, 16, 8, 256, 1, 0, 4096), (0, 100, 28, 4, 128, 0, 0, 0)]:
        assert L.hcp_plan_fwd_split(*args, ctypes.addressof(w), ctypes.addressof(nb)) == 0
        assert (w.value, nb.value) == (0, 0)
    # one chunk of a long prompt is cut, and the workspace holds its partials
    pt = L.hcp_plan_fwd_split(512, 32768, 28, 4, 128, 1, 32256, 0, ctypes.addressof(w),
                              ctypes.addressof(nb))
    np_ = -(-512 // pt)
    assert pt > 0 and w.value == 0 and nb.value == 4 * np_ * 28 * 128 * 129 * 4
    assert L.hcp_plan_fwd_split(4, 4, 28, 3, 128, 0, 0, 0, ctypes.addressof(w),
                                ctypes.addressof(nb)) == _lib.HCP_EINVAL
