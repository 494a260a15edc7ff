"""The framework's work as a serving program gives it, one case per kind of call.

A case is a dict of plain numbers and texts; its "kind" picks the path:

* ``ring``     one layer of a ring prefill on the kernel contract: the peer chunk non-causal, the
               local chunk causal, merged by LSE (``ring_attn_with_lse`` + ``ring_attn_merged``, or
               the three-call form with ``merge_attn_states``), or a windowed local pass alone.
* ``forward``  ``HcpRingAttentionImpl.forward`` over the layers of one engine step: prefill chunks,
               decode rows and mixtures of both over the paged cache, with or without staged peer
               prefixes.  Every pass is a step of its own: a new metadata object, as the engine's
               metadata builder makes one per step.
* ``hop``      one hop of the decode ring on a node (``RingDecodeNode.accumulate``).
* ``write``    the paged KV write of a step (``reshape_and_cache``).

Attention shapes are those of this repository's benchmark and tests: 28 / 4 heads x 128, 14 / 2 x 64,
64 / 8 x 128 and 16 / 8 x 256.  Values are N(0, 1) with a few K channels scaled up (logit outliers).
"""

from __future__ import annotations

import itertools
import math
import random
import types
import weakref

import torch

from hcp_vllm_plugin_amd import merge_attn_states, ring_attn_merged, ring_attn_with_lse
from hcp_vllm_plugin_amd import ring_backend as rb
from hcp_vllm_plugin_amd.kv_cache import reshape_and_cache
from hcp_vllm_plugin_amd.ring_decode import RING_NODES, RingDecodeNode

SHAPES = {"28/4x128": (28, 4, 128), "14/2x64": (14, 2, 64),
          "64/8x128": (64, 8, 128), "16/8x256": (16, 8, 256)}
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
LARGEST_FLOPS = 4.2e12  # a drawn case stays below the largest listed one
LARGEST_BYTES = 1.78e10
_ids = itertools.count()


def _ring(name, shape, dtype, local, peer, offset=0, window=0, merge="fused"):
    return {"name": name, "kind": "ring", "shape": shape, "dtype": dtype, "local": local,
            "peer": peer, "offset": offset, "window": window, "merge": merge}


def _forward(name, shape="28/4x128", dtype="bf16", layout="v031", block=16, layers=1,
             prefills=0, new_lo=1, new_hi=1, before_lo=0, before_hi=0,
             decodes=0, ctx_lo=1, ctx_hi=1, peer_lo=0, peer_hi=0):
    return {"name": name, "kind": "forward", "shape": shape, "dtype": dtype, "layout": layout,
            "block": block, "layers": layers, "prefills": prefills, "new_lo": new_lo,
            "new_hi": new_hi, "before_lo": before_lo, "before_hi": before_hi, "decodes": decodes,
            "ctx_lo": ctx_lo, "ctx_hi": ctx_hi, "peer_lo": peer_lo, "peer_hi": peer_hi}


def listed():
    return [
        # the headline ring prefill step of a 16k prompt split over two workers
        _ring("ring-8k", "28/4x128", "bf16", 8192, 8192),
        # a short prompt: the smallest ring step, in the reference's three-call form
        _ring("ring-256", "28/4x128", "fp16", 256, 256, merge="calls"),
        # the small model of the reference's probes, ragged chunks, three-call form
        _ring("ring-d64", "14/2x64", "fp16", 3001, 5003, merge="calls"),
        # a sliding-window layer of a head_dim 256 model
        _ring("window-d256", "16/8x256", "bf16", 8192, 0, window=4096),
        # chunked prefill: a 512-token chunk near the end of a 32k prompt
        _forward("chunk-512", layers=2, prefills=1, new_lo=512, new_hi=512,
                 before_lo=32256, before_hi=32256),
        # a prefill batch of 16 ragged requests whose prefixes are staged peer chunks
        _forward("prefill-16", prefills=16, new_lo=512, new_hi=4096, peer_lo=1024, peer_hi=16384),
        # continuous batching: one prefill chunk next to 32 decoding requests
        _forward("mixed-33", layers=2, prefills=1, new_lo=512, new_hi=512, before_lo=3584,
                 before_hi=3584, decodes=32, ctx_lo=512, ctx_hi=8192),
        # one user's decode step at a short context: the smallest forward
        _forward("decode-1", layers=4, decodes=1, ctx_lo=2000, ctx_hi=2000),
        # an ordinary decode batch over the paged cache
        _forward("decode-16", dtype="fp16", layout="v023", layers=4, decodes=16, ctx_lo=1024,
                 ctx_hi=8192),
        # the headline decode batch: 32k staged prefixes, paged local keys
        _forward("decode-64", layers=4, decodes=64, ctx_lo=512, ctx_hi=2048, peer_lo=32768,
                 peer_hi=32768),
        # one decode-ring hop: a 32k chunk snapshot and 512 growth tokens
        {"name": "hop-32k", "kind": "hop", "shape": "28/4x128", "dtype": "bf16", "chunk": 32768,
         "growth": 512},
        # the paged KV write of an 8k prefill step
        {"name": "write-8k", "kind": "write", "shape": "28/4x128", "dtype": "bf16",
         "layout": "v031", "block": 16, "tokens": 8192},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    while True:
        kind = rng.choice(["ring", "ring", "window", "chunk", "prefill", "mixed", "decode",
                           "decode", "staged", "hop", "write"])
        shape = rng.choice(list(SHAPES))
        dtype = rng.choice(list(DTYPES))
        layout, block = rng.choice(["v031", "v023"]), rng.choice([16, 16, 32, 64])
        paged = dict(shape=shape, dtype=dtype, layout=layout, block=block)
        if kind == "ring":
            c = _ring("", shape, dtype, _log(rng, 64, 8192), _log(rng, 64, 8192),
                      offset=rng.choice([0, 0, _log(rng, 1, 8192)]),
                      merge=rng.choice(["fused", "calls"]))
        elif kind == "window":
            c = _ring("", shape, dtype, _log(rng, 256, 8192), 0, offset=rng.choice([0, 1000]),
                      window=_log(rng, 128, 4096))
        elif kind == "chunk":
            new, before = _log(rng, 16, 2048), _log(rng, 512, 65536)
            c = _forward("", layers=2, prefills=1, new_lo=new, new_hi=new, before_lo=before,
                         before_hi=before, **paged)
        elif kind == "prefill":
            hi, peer = _log(rng, 64, 4096), rng.choice([0, _log(rng, 256, 16384)])
            c = _forward("", prefills=rng.randint(2, 16), new_lo=max(1, hi // 8), new_hi=hi,
                         peer_lo=peer // 16, peer_hi=peer, **paged)
        elif kind == "mixed":
            new, ctx = _log(rng, 64, 2048), _log(rng, 512, 16384)
            c = _forward("", layers=2, prefills=rng.randint(1, 3), new_lo=max(1, new // 2),
                         new_hi=new, before_lo=0, before_hi=_log(rng, 1, 8192),
                         decodes=_log(rng, 1, 64), ctx_lo=max(1, ctx // 16), ctx_hi=ctx, **paged)
        elif kind == "decode":
            ctx = _log(rng, 128, 32768)
            c = _forward("", layers=4, decodes=_log(rng, 1, 128), ctx_lo=max(1, ctx // 8),
                         ctx_hi=ctx, **paged)
        elif kind == "staged":
            ctx, peer = _log(rng, 64, 4096), _log(rng, 512, 32768)
            c = _forward("", layers=4, decodes=_log(rng, 1, 64), ctx_lo=max(1, ctx // 4),
                         ctx_hi=ctx, peer_lo=peer, peer_hi=peer, **paged)
        elif kind == "hop":
            c = {"kind": "hop", "shape": shape, "dtype": dtype, "chunk": _log(rng, 512, 65536),
                 "growth": rng.choice([0, _log(rng, 1, 2048)])}
        else:
            c = {"kind": "write", "shape": shape, "dtype": dtype, "layout": layout,
                 "block": block, "tokens": _log(rng, 1, 32768)}
        c.pop("name", None)
        w = work(c)
        if w["flops"] <= LARGEST_FLOPS and w["bytes"] <= LARGEST_BYTES:
            return c


# -- sizes --------------------------------------------------------------------
def _requests(case):
    """(new tokens, peer prefix, local keys) of each request, the same for every
    seed: the keys a query sees are the prefix and the local ones up to itself."""
    r = random.Random("%(new_lo)d %(new_hi)d %(before_lo)d %(before_hi)d %(ctx_lo)d %(ctx_hi)d "
                      "%(peer_lo)d %(peer_hi)d" % case)
    bs, out = case["block"], []

    def peer():
        n = r.randint(case["peer_lo"], case["peer_hi"])
        return max(bs, n // bs * bs) if n else 0  # prefixes are whole blocks

    for _ in range(case["prefills"]):
        new = r.randint(case["new_lo"], case["new_hi"])
        out.append((new, peer(), new + r.randint(case["before_lo"], case["before_hi"])))
    for _ in range(case["decodes"]):
        out.append((1, peer(), r.randint(case["ctx_lo"], case["ctx_hi"])))
    return out


def _pairs(tq, tk, off, window=0):
    """Visible (query, key) pairs of a causal pass."""
    hi = torch.clamp(torch.arange(tq, dtype=torch.int64) + off + 1, max=tk)
    lo = torch.clamp(torch.arange(tq, dtype=torch.int64) + off + 1 - window, min=0) if window else 0
    return int((hi - lo).sum())


def work(case):
    h, hkv, d = SHAPES[case["shape"]]
    if case["kind"] == "ring":
        t, off, p = case["local"], case["offset"], case["peer"]
        pairs = _pairs(t, t + off, off, case["window"]) + t * p
        keys = t + off + p
        return {"bytes": (2 * t * h + 2 * keys * hkv) * d * 2 + t * h * 4,
                "flops": 4 * d * h * pairs}
    if case["kind"] == "forward":
        reqs = _requests(case)
        pairs = sum(_pairs(n, loc, loc - n) + n * p for n, p, loc in reqs)
        rows, keys = sum(n for n, _, _ in reqs), sum(p + loc for _, p, loc in reqs)
        return {"bytes": case["layers"] * (2 * rows * h + 2 * keys * hkv) * d * 2,
                "flops": case["layers"] * 4 * d * h * pairs}
    if case["kind"] == "hop":
        keys = case["chunk"] + case["growth"]
        return {"bytes": (3 * h + 2 * keys * hkv) * d * 2 + 2 * h * 4, "flops": 4 * d * h * keys}
    return {"bytes": case["tokens"] * (4 * hkv * d * 2 + 8), "flops": 0}


# -- inputs -------------------------------------------------------------------
class _Draw:
    """Seeded values on the GPU: N(0, 1) rounded to the case's dtype, four K
    channels scaled by 8 as the outlier channels of trained models are."""

    def __init__(self, case, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)
        self.dtype = DTYPES[case["dtype"]]
        d = SHAPES[case["shape"]][2]
        self.ch = torch.randperm(d, device="cuda", generator=self.gen)[:4]

    def randn(self, *shape):
        return torch.empty(*shape, dtype=self.dtype, device="cuda").normal_(generator=self.gen)

    def keys(self, *shape):
        k = self.randn(*shape)
        k[..., self.ch] *= 8
        return k


class _State:
    """A case's inputs; what it registered with the backend goes with it."""


def _drop(chunks, first_blocks):
    for c in chunks:
        rb.drop_chunk_kv(c)
    for b in first_blocks:
        rb.unmap_request_peer(b)


def _prepare_forward(case, seed, d):
    h, hkv, dim = SHAPES[case["shape"]]
    reqs, bs, n_id = _requests(case), case["block"], next(_ids)
    s = _State()
    need = [-(-loc // bs) for _, _, loc in reqs]  # blocks of the local keys
    nb = sum(need) + 4
    perm = torch.randperm(nb, device="cuda", generator=d.gen).to(torch.int32)
    bt = torch.zeros(len(reqs), max(p // bs + n for (_, p, _), n in zip(reqs, need)),
                     dtype=torch.int32, device="cuda")
    at = 0
    for r, ((_, p, _), n) in enumerate(zip(reqs, need)):
        bt[r, p // bs:p // bs + n] = perm[at:at + n]
        at += n
    s.layers = [types.SimpleNamespace(layer_name="model.layers.%d.self_attn.attn" % i)
                for i in range(case["layers"])]
    s.q, s.caches, s.peers, chunks, firsts = [], [], [], [], []
    rows = sum(n for n, _, _ in reqs)
    for layer in s.layers:
        s.q.append(d.randn(rows, h, dim))
        if case["layout"] == "v031":
            c = d.randn(nb, hkv, bs, 2 * dim)
            c[..., d.ch] *= 8
        else:
            c = d.randn(nb, 2, bs, hkv, dim)
            c[:, 0, ..., d.ch] *= 8
        s.caches.append(c)
        peers = []
        for r, (_, p, _) in enumerate(reqs):
            # a staged prefix as the backend stores it, head-major
            kv = (d.keys(hkv, p, dim).permute(1, 0, 2), d.randn(hkv, p, dim).permute(1, 0, 2)) \
                if p else None
            peers.append(kv)
            if p:
                rb.stage_peer_kv("perf%d-req%d" % (n_id, r), layer.layer_name, *kv)
        s.peers.append(peers)
    for r, (_, p, _) in enumerate(reqs):
        if p:  # the prefix's pool slots are never read: the first names the request
            first = (1 << 24) + n_id * 1024 + r
            bt[r, 0] = first
            chunks.append("perf%d-req%d" % (n_id, r))
            firsts.append(first)
            rb.map_request_peer(first, [chunks[-1]])
    if firsts:
        weakref.finalize(s, _drop, chunks, firsts)
    s.bt = bt
    qsl = [0]
    for n, _, _ in reqs:
        qsl.append(qsl[-1] + n)
    s.rows = rows
    s.qsl = torch.tensor(qsl, dtype=torch.int32, device="cuda")
    s.lens = torch.tensor([p + loc for _, p, loc in reqs], dtype=torch.int32, device="cuda")
    s.impl = rb.HcpRingAttentionImpl(h, dim, 1 / math.sqrt(dim), hkv)
    s.out = [torch.empty_like(q) for q in s.q]
    return s


def prepare(case, seed):
    h, hkv, dim = SHAPES[case["shape"]]
    d = _Draw(case, seed)
    if case["kind"] == "forward":
        s = _prepare_forward(case, seed, d)
    elif case["kind"] == "ring":
        s = _State()
        t, tk, p = case["local"], case["local"] + case["offset"], case["peer"]
        s.q = d.randn(t, h, dim)
        s.k, s.v = d.keys(tk, hkv, dim), d.randn(tk, hkv, dim)
        s.pk, s.pv = d.keys(p, hkv, dim), d.randn(p, hkv, dim)
    elif case["kind"] == "hop":
        s = _State()
        s.k, s.v = d.keys(case["chunk"], hkv, dim), d.randn(case["chunk"], hkv, dim)
        s.gk, s.gv = d.keys(case["growth"], hkv, dim), d.randn(case["growth"], hkv, dim)
        s.q, s.o = d.randn(1, h, dim), d.randn(1, h, dim)
        # the accumulator of the hops before: as many keys again
        s.lse = torch.empty(h, 1, device="cuda").normal_(generator=d.gen) \
            + math.log(case["chunk"]) + 1.0
        s.node = RingDecodeNode("", ["chunk"], 0, dtype=d.dtype, background=False)
        RING_NODES.remove(s.node)  # the registry would keep every state's keys
        s.node.add_chunk("chunk", "layer", s.k, s.v)
        if case["growth"]:
            s.node.append_growth("req", "layer", s.gk, s.gv)
        s.node.mark_ready()
    else:
        s = _State()
        n, bs = case["tokens"], case["block"]
        nb = -(-n // bs) + -(-n // (4 * bs)) + 1
        s.key, s.value = d.randn(n, hkv, dim), d.randn(n, hkv, dim)
        # a prefill writes whole blocks: runs of neighbouring slots
        s.slots = torch.randperm(nb, device="cuda", generator=d.gen)[:-(-n // bs)]
        s.slots = (s.slots[:, None] * bs + torch.arange(bs, device="cuda")).reshape(-1)[:n] \
            .contiguous()
        shape = (nb, hkv, bs, 2 * dim) if case["layout"] == "v031" else (nb, 2, bs, hkv, dim)
        s.cache = torch.zeros(*shape, dtype=d.dtype, device="cuda")
    s.case = case
    return s


# -- one pass -----------------------------------------------------------------
def run(s):
    case = s.case
    if case["kind"] == "forward":
        meta = types.SimpleNamespace(num_actual_tokens=s.rows, query_start_loc=s.qsl,
                                     seq_lens=s.lens, block_table=s.bt)
        return [s.impl.forward(layer, q, None, None, cache, meta, out)
                for layer, q, cache, out in zip(s.layers, s.q, s.caches, s.out)]
    if case["kind"] == "hop":
        return s.node.accumulate(s.q, s.o, s.lse, 1 / math.sqrt(s.q.shape[2]), "layer", "req")
    if case["kind"] == "write":
        reshape_and_cache(s.key, s.value, s.cache, s.slots)
        return s.cache
    scale = 1 / math.sqrt(s.q.shape[2])
    if not case["peer"]:
        return ring_attn_with_lse(s.q, s.k, s.v, scale, case["offset"], case["window"] or None)
    lse = torch.empty(s.q.shape[1], s.q.shape[0], device="cuda")
    if case["merge"] == "fused":
        o, l = ring_attn_with_lse(s.q, s.pk, s.pv, scale, None)
        out = ring_attn_merged(s.q, s.k, s.v, scale, case["offset"], o, l, output_lse=lse)
        return out, lse
    o, l = ring_attn_with_lse(s.q, s.k, s.v, scale, case["offset"])
    po, pl = ring_attn_with_lse(s.q, s.pk, s.pv, scale, None)
    out = torch.empty_like(o)
    merge_attn_states(out, po, pl, o, l, lse)
    return out, lse


def tolerance(case):
    """The 16-bit output's own rounding and that of P before the PV product: the
    path is 1.6e-3 to 2.7e-3 (bf16) and 2.2e-4 to 3.4e-4 (fp16) from ``exact``
    (an LSE 6e-8); four times the largest."""
    if case["kind"] == "write":
        return "exact"
    if case["dtype"] == "bf16":
        return {"rel": 1.1e-2, "max": 8e-2}
    return {"rel": 1.4e-3, "max": 1e-2}


# -- the same in 64 bits ------------------------------------------------------
def _attend(q, k, v, scale, off=None, window=0, skip=0):
    """(out, lse) of q [T, H, D] over k, v [N, Hkv, D] in float64; with ``off``
    key j >= skip is visible to row i iff j - skip <= off + i (and, windowed,
    j - skip > off + i - window); keys before ``skip`` always are."""
    t, h, d = q.shape
    n, hkv, _ = k.shape
    g = h // hkv
    out = torch.zeros(t, h, d, dtype=torch.float64, device=q.device)
    lse = torch.full((h, t), float("-inf"), dtype=torch.float64, device=q.device)
    step = max(1, min(t, (1 << 27) // max(n, 1)))
    pos = torch.arange(n, device=q.device) - skip
    for kh in range(hkv):
        kt, vv = k[:, kh].double().t().contiguous(), v[:, kh].double()
        for h0 in range(kh * g, kh * g + g):
            for a in range(0, t, step):
                b = min(t, a + step)
                sc = (q[a:b, h0].double() @ kt) * scale
                if off is not None:
                    last = off + torch.arange(a, b, device=q.device)[:, None]
                    hide = pos > last
                    if window:
                        hide |= pos <= last - window
                    sc.masked_fill_(hide, float("-inf"))
                l = torch.logsumexp(sc, 1)
                lse[h0, a:b] = l
                out[a:b, h0] = sc.sub_(l[:, None]).exp_() @ vv
    return out, lse


def exact(case, seed):
    s = prepare(case, seed)
    if case["kind"] == "write":
        return None
    scale = 1 / math.sqrt(s.q[0].shape[2] if case["kind"] == "forward" else s.q.shape[2])
    if case["kind"] == "ring":
        k, v = torch.cat([s.pk, s.k]), torch.cat([s.pv, s.v])
        return _attend(s.q, k, v, scale, case["offset"], case["window"], skip=case["peer"])
    if case["kind"] == "hop":
        o, l = _attend(s.q, torch.cat([s.k, s.gk]), torch.cat([s.v, s.gv]), scale)
        la = s.lse.double()
        m = torch.logaddexp(la, l)
        wa, w = torch.exp(la - m).t()[..., None], torch.exp(l - m).t()[..., None]
        return s.o.double() * wa + o * w, m
    outs = []
    bs, qsl, reqs = case["block"], s.qsl.tolist(), _requests(case)
    for q, cache, peers in zip(s.q, s.caches, s.peers):
        out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
        for r, (new, p, loc) in enumerate(reqs):
            ids = s.bt[r, p // bs:p // bs + -(-loc // bs)].long()
            if case["layout"] == "v031":
                kv = cache[ids].permute(0, 2, 1, 3).reshape(-1, cache.shape[1], cache.shape[3])
                k, v = kv[:loc].chunk(2, -1)
            else:
                k, v = (cache[ids, i].reshape(-1, *cache.shape[3:])[:loc] for i in (0, 1))
            if p:
                k, v = torch.cat([peers[r][0], k]), torch.cat([peers[r][1], v])
            a, b = qsl[r], qsl[r + 1]
            out[a:b] = _attend(q[a:b], k, v, scale, loc - new, skip=p)[0]
        outs.append(out)
    return outs
