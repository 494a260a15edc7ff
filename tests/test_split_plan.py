"""The split planners on the CPU: every (query block, tile) of a prefill batch is in
exactly one piece, slots are used once, and a launch that fills the machine is
left whole (``hcp_plan_varlen_split``, ``hcp_plan_fwd_split``); every key of a
decode batch is in exactly one record (``hcp_plan_decode_lists``)."""

import ctypes

import numpy as np
import pytest

from hcp_vllm_plugin_amd import _lib
from hcp_vllm_plugin_amd.varlen import ENTRY_DTYPE, WORK_DTYPE

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


def _lists(lens, seqs, num_seqs, workgroups, split_tokens=0):
    n = len(lens)
    a = np.zeros(max(n, 1), dtype=ENTRY_DTYPE)
    a["q_len"], a["q_start"][:n], a["len"][:n] = 1, seqs, lens
    cap = n + workgroups + (sum(-(-x // split_tokens) for x in lens) if split_tokens else 0)
    works = np.zeros(max(cap, 1), dtype=WORK_DTYPE)
    entry, starts = np.zeros(max(cap, 1), np.int32), np.zeros(num_seqs + 1, np.int32)
    seq, m = np.asarray(list(seqs) or [0], np.int32), ctypes.c_int32(0)
    L = _lib.lib()
    rc = L.hcp_plan_decode_lists(a.ctypes.data, n, seq.ctypes.data, num_seqs, workgroups,
                                 split_tokens, works.ctypes.data, entry.ctypes.data, cap,
                                 starts.ctypes.data, ctypes.addressof(m))
    _lib.check(rc, "hcp_plan_decode_lists")
    return works[:rc], entry[:rc], starts, m.value


@pytest.mark.parametrize("workgroups,split", [(64, 0), (1, 0), (7, 0), (256, 0), (0, 64), (0, 1000)])
@pytest.mark.parametrize("lens,seqs,num_seqs", [
    ([2000], [0], 1), ([1], [0], 1), ([32768, 512], [0, 0], 1), ([], [], 3),
    ([5000, 0, 31, 33, 8192, 64], [0, 0, 1, 3, 3, 4], 6), ([100] * 300, range(300), 300),
    ([513, 2048, 700, 1999] * 16, range(64), 64),
])
def test_decode_lists_cover_every_key_once(lens, seqs, num_seqs, workgroups, split):
    works, entry, starts, wgs = _lists(lens, seqs, num_seqs, workgroups, split)
    assert wgs <= (workgroups or len(works))
    # every record is reached from exactly one workgroup's list
    seen, loads = set(), []
    for w in range(wgs):
        load, j = 0, w
        while j >= 0:
            assert j not in seen
            seen.add(j)
            load += 8 - (int(works[j]["key_begin"]) - int(works[j]["key_end"])) // 32
            j = int(works[j]["next"])
        loads.append(load)
    assert seen == set(range(len(works)))
    # slots: one each, in sequence order; key ranges: each entry cut end to end
    by_slot = np.argsort(works["slot"])
    assert (works["slot"][by_slot] == np.arange(len(works))).all()
    pos = [0] * len(lens)
    for j in by_slot:
        e, w = int(entry[j]), works[j]
        assert w["e"]["q_start"] == list(seqs)[e] and w["e"]["len"] == lens[e]
        assert w["key_begin"] == pos[e] < w["key_end"]
        pos[e] = int(w["key_end"])
        assert starts[list(seqs)[e]] <= w["slot"] < starts[list(seqs)[e] + 1]
        if split:
            assert w["key_end"] - w["key_begin"] <= split
    assert pos == list(lens) and starts[0] == 0 and starts[-1] == len(works)
    if not split and len(works):  # no workgroup far above an even share
        even = (sum(-(-x // 32) for x in lens) + 8 * len(works)) / workgroups
        assert max(loads) <= even + 8 + 16


def test_decode_lists_refuse_bad_input():
    L = _lib.lib()
    a = np.zeros(2, dtype=ENTRY_DTYPE)
    a["q_len"], a["len"] = 1, 1000
    works, starts = np.zeros(4, dtype=WORK_DTYPE), np.zeros(3, np.int32)
    m = ctypes.c_int32(0)

    def call(seq, ns=2, wgs=64, st=0, cap=4):
        s = np.asarray(seq, np.int32)
        return L.hcp_plan_decode_lists(a.ctypes.data, 2, s.ctypes.data, ns, wgs, st,
                                       works.ctypes.data, 0, cap, starts.ctypes.data,
                                       ctypes.addressof(m))

    assert call([1, 0]) == call([0, 2]) == call([0, 1], wgs=0) == _lib.HCP_EINVAL
    assert call([0, 1], st=64) == _lib.HCP_EINVAL
    assert call([0, 1], cap=1) == _lib.HCP_EWORKSPACE
    a["q_len"] = 2
    assert call([0, 1]) == _lib.HCP_EINVAL
