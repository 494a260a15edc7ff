"""What planning a launch costs the host, on the CPU: the planners' own calls
counted, and the plans of equal batches equal."""

import ctypes

import numpy as np
import pytest
import torch

from hcp_vllm_plugin_amd import varlen as V

CPU = torch.device("cpu")


@pytest.fixture
def uploads(monkeypatch):
    """Byte counts of what each plan uploads, and the blocks themselves."""
    got = []

    def upload(arrays, device):
        offs, raw = [], b""  # (addresses: offsets in the block)
        for a in arrays:
            offs.append(len(raw))
            n, addr = V._nbytes_addr(a)
            raw += ctypes.string_at(addr, n)
            raw += b"\0" * (-len(raw) % 256)
        got.append(raw)
        return None, offs

    monkeypatch.setattr(V, "_upload", upload)
    return got


def _seg(n):
    s = V.KvSegment()
    s.k_addr = s.v_addr = 4096
    s.stride_tok, s.stride_head, s.len = 128, n * 128, n
    return s


@pytest.mark.parametrize("rows", [None, [7, 3]])
@pytest.mark.parametrize("split", [None, 64, 1000])
def test_decode_plans_of_both_forms_agree(uploads, rows, split):
    """Segments as objects and the same as an entry array: the same records,
    where the launch arguments say."""
    segs = [[_seg(5000), _seg(33)], [_seg(700)]]
    a = V.DecodeBatch(segs, 28, 4, 128, CPU, split, rows=rows)
    ent = np.zeros(3, dtype=V.ENTRY_DTYPE)
    for i, (s, seg) in enumerate([(0, segs[0][0]), (0, segs[0][1]), (1, segs[1][0])]):
        e = V.make_entry(s if rows is None else rows[s], 1, seg, 0)
        ent[i] = np.frombuffer(e, dtype=V.ENTRY_DTYPE)[0]
    b = V.DecodeBatch.from_entries(ent, 28, 4, 128, CPU, split, rows=rows, num_seqs=2,
                                   entry_seq=np.array([0, 0, 1], np.int32))
    assert a.split_tokens == b.split_tokens and a.num_splits == b.num_splits == a._args.num_works
    raw, other = uploads
    works = np.frombuffer(raw, V.WORK_DTYPE, a.num_splits, a._args.works)
    same = np.frombuffer(other, V.WORK_DTYPE, a.num_splits, b._args.works)
    starts = np.frombuffer(raw, np.int32, 3, a._args.seq_partial_start)
    assert (works == same).all() and starts[0] == 0 and starts[2] == a.num_splits
    assert int((works["key_end"] - works["key_begin"]).sum()) == 5733
    if rows is None:
        assert a._args.seq_rows == 0
    else:
        assert np.frombuffer(raw, np.int32, 2, a._args.seq_rows).tolist() == rows
    with pytest.raises(ValueError, match="one row per sequence"):
        V.DecodeBatch(segs, 28, 4, 128, CPU, split, rows=[1, 2, 3])


def test_decode_plan_is_one_host_block(uploads, monkeypatch):
    """... not an array each for records, starts, rows and their conversions:
    a hop plans again after every growth append."""
    made = []
    empty = np.empty
    monkeypatch.setattr(np, "empty", lambda *a, **k: made.append(a) or empty(*a, **k))
    V.DecodeBatch([[_seg(32768), _seg(512)]], 28, 4, 128, CPU)
    assert len(made) == 1


@pytest.mark.parametrize("causal,window", [(True, None), (True, 300), (False, None)])
@pytest.mark.parametrize("paged", [False, True])
def test_launches_of_equal_sizes_share_a_cut(uploads, monkeypatch, causal, window, paged):
    """The search for the KV split runs once for the layers of a step, at other
    addresses too; other sizes, offsets, windows or heads get their own."""
    V._varlen_cut.cache_clear()
    L = V._lib.lib()
    calls, plan = [], L.hcp_plan_varlen_split
    monkeypatch.setattr(L, "hcp_plan_varlen_split", lambda *a: calls.append(a) or plan(*a))

    def launch(addr, keys=32768, heads=(28, 4, 128), new=512, win=window):
        e = np.zeros(2, dtype=V.ENTRY_DTYPE)
        e["q_len"], e["q_start"], e["len"] = [new, 3], [0, new], [keys, 700]
        e["causal_offset"] = e["len"] - e["q_len"] if causal else 0
        e["k_addr"] = e["v_addr"] = addr
        e["stride_tok"], e["stride_head"] = 512, 128
        if paged:
            e["block_table"], e["stride_block"], e["block_size"] = addr, 8192, 16
        return V.VarlenLaunch(e, causal, paged, CPU, heads=heads, window=win)

    first = launch(4096)
    assert len(calls) == 1
    for i in range(3):
        same = launch(8192 * (i + 1))
        assert same._split == first._split
    assert len(calls) == 1
    if window is None:  # 512 x 32768 at 28 heads is cut, whatever the form
        assert first._split is not None and first._split["pieces"] > 2 * 4
        up = uploads[-1]
        assert first._split["pieces"] * 16 + first._split["units"] * 16 < len(up)
    launch(4096, keys=30000), launch(4096, heads=(14, 2, 64)), launch(4096, new=500)
    launch(4096, win=900)
    assert len(calls) == (5 if causal else 4)  # a window is nothing to a launch without a mask
    assert V._varlen_cut.cache_info().maxsize == 64


def test_a_launchs_arguments_are_its_own(uploads):
    """(The addresses of the uploaded records go into them.)"""
    e = np.zeros(1, dtype=V.ENTRY_DTYPE)
    e["q_len"], e["len"], e["stride_tok"], e["stride_head"] = 64, 8192, 512, 128
    a = V.VarlenLaunch(e, False, False, CPU, heads=(28, 4, 128))
    b = V.VarlenLaunch(e, False, False, CPU, heads=(28, 4, 128))
    a._split["ptrs"] = "a"
    assert b._split["ptrs"] != "a" and a._split is not b._split


def test_rebound_chunks_follow_the_entries(uploads):
    """Row i of a rebind goes to the records of the i-th contiguous entry and
    to no other, whatever a rebind before it was given; one with another
    number of rows is refused."""
    ent = np.zeros(5, dtype=V.ENTRY_DTYPE)
    ent["q_len"], ent["len"] = 1, [3000, 900, 5000, 64, 7000]
    ent["block_table"], ent["k_addr"] = [4096, 0, 0, 8192, 0], [1, 2, 3, 4, 5]
    seq = np.array([0, 0, 1, 2, 2], np.int32)
    plan = V.DecodeBatch.from_entries(ent, 28, 4, 128, CPU, entry_seq=seq, num_seqs=3)
    at0 = plan._args.works
    for base in (100, 200):
        rows = (np.arange(12, dtype=np.uint64) + base).reshape(3, 4)
        got = plan.rebind_chunks(rows)
        works = np.frombuffer(uploads[-1], V.WORK_DTYPE, plan.num_splits, got._args.works)
        before = np.frombuffer(uploads[0], V.WORK_DTYPE, plan.num_splits, at0)
        for w, old in zip(works, before):
            at = {2: 0, 3: 1, 5: 2}.get(int(old["e"]["k_addr"]))
            fields = [int(w["e"][f]) for f in ("k_addr", "v_addr", "stride_tok", "stride_head")]
            assert fields == ([int(old["e"]["k_addr"]), 0, 0, 0] if at is None
                              else rows[at].tolist())
            assert w["key_begin"] == old["key_begin"] and w["next"] == old["next"]
        plan = got  # a copy inherits what it memoised
    for wrong in (rows[:2], np.zeros((4, 4), np.uint64)):
        with pytest.raises(ValueError, match="one row per contiguous entry"):
            plan.rebind_chunks(wrong)
