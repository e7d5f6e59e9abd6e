"""The work whose speed is measured: what a program that serves a model from
this KV cache has it do, over the range of sizes such programs have.

A pass goes through the public entry points of `emelk` only.  The kinds:

  decode    one token per sequence: store it and attend to the history
            (decode_append), for every layer of the case.  More than one layer
            is one HIP graph that the program captured once and replays per
            step, as a serving loop does; a single layer is a plain call.
  flash     the same on one contiguous cache without a block table
            (decode_contiguous), the layout a single sequence has.
  executor  BatchDecoder: begin_step, then every layer (norm, RoPE, store,
            attention), launched call by call.  The pass takes its tokens back
            (rollback_slots) as a program does that rejects drafted tokens, so
            every pass starts from the same history.
  chunk     several tokens per sequence of one layer: store them (append), then
            causal attention over the prefix and the chunk (prefill_chunk).
  rope      the step between the projections and the attention for a prompt
            chunk: norms, RoPE, store (qkv_rope_append).
  gather    the cached tokens of every layer to dense rows (gather), as a
            program does that saves a session.
  compact   the page moves of an eviction applied to every layer
            (copy_blocks).

Sizes are those of the benchmark and the tests (Qwen3-0.6B, Llama-3.2-1B,
Llama-3-8B and Gemma-4 shapes), K, V and Q are N(0, 1); q8_0 caches have 1% of
the values scaled by 20, as outliers.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "emel.cpp_amd"))
import emelk  # noqa: E402

DEV = "cuda"


# ---- the cases ----------------------------------------------------------------

def _shape(heads, kv_heads, dim, page, kv):
    return {"heads": heads, "kv_heads": kv_heads, "dim": dim, "page": page, "kv": kv}


def listed():
    return [
        # one user's chat on a small model, a step of all 28 layers: the
        # smallest launches, where latency is everything
        {"name": "flash-0.6b-1x513", "kind": "flash", "layers": 28, "seqs": 1, "len_min": 513,
         "len_max": 513, "capacity": 1024, **_shape(16, 8, 128, 1024, "f16")},
        # a small server: 16 users with contexts of different lengths, a step
        # of all 16 layers
        {"name": "decode-1b-16xragged", "kind": "decode", "layers": 16, "seqs": 16,
         "len_min": 1025, "len_max": 4097, **_shape(32, 8, 64, 16, "f16")},
        # a full server, one layer of the step: 2 GB of K and V
        {"name": "decode-8b-64x8k", "kind": "decode", "layers": 1, "seqs": 64, "len_min": 8193,
         "len_max": 8193, **_shape(32, 8, 128, 32, "f16")},
        # long contexts on a quantized cache, one layer of the step
        {"name": "decode-8b-q8-32x16k", "kind": "decode", "layers": 1, "seqs": 32,
         "len_min": 16385, "len_max": 16385, **_shape(32, 8, 128, 32, "q8_0")},
        # the step executor, call by call, with head norms and halved-pair RoPE
        {"name": "executor-0.6b-8xragged", "kind": "executor", "layers": 28, "seqs": 8,
         "tokens": 1, "len_min": 200, "len_max": 1500, **_shape(16, 8, 128, 16, "f16")},
        # drafted tokens of four users checked in one call
        {"name": "chunk-8b-4x6-draft", "kind": "chunk", "seqs": 4, "tokens": 6, "len_min": 2000,
         "len_max": 6000, **_shape(32, 8, 128, 32, "f16")},
        # one user's prompt: a 512-token chunk of a single sequence, 256-wide
        # heads (eight query heads on one KV head)
        {"name": "chunk-gemma-1x512", "kind": "chunk", "seqs": 1, "tokens": 512, "len_min": 2048,
         "len_max": 2048, **_shape(8, 1, 256, 32, "f16")},
        # prompts of eight users in chunks of 512
        {"name": "chunk-8b-8x512", "kind": "chunk", "seqs": 8, "tokens": 512, "len_min": 4096,
         "len_max": 4096, **_shape(32, 8, 128, 32, "f16")},
        # the same on a quantized cache
        {"name": "chunk-8b-q8-8x512", "kind": "chunk", "seqs": 8, "tokens": 512, "len_min": 4096,
         "len_max": 4096, **_shape(32, 8, 128, 32, "q8_0")},
        # the rows of a prompt chunk with head norms, on their way into the cache
        {"name": "rope-0.6b-8x512-norm", "kind": "rope", "seqs": 8, "tokens": 512, "len_min": 100,
         "len_max": 4000, "norm": True, "v_norm": False, "neox": True,
         **_shape(16, 8, 128, 16, "f16")},
        # a quantized session saved
        {"name": "gather-8b-q8-8x4k", "kind": "gather", "layers": 4, "seqs": 8, "len_min": 3000,
         "len_max": 4096, **_shape(32, 8, 128, 32, "q8_0")},
        # a quarter of eight sequences' pages evicted, the rest moved together
        {"name": "compact-8b-8x4k", "kind": "compact", "layers": 32, "seqs": 8, "len_min": 4608,
         "len_max": 4608, **_shape(32, 8, 128, 32, "f16")},
    ]


_HEADS = [(16, 8, 128), (32, 8, 64), (32, 8, 128), (8, 8, 64), (64, 8, 128), (8, 2, 128),
          (8, 1, 256), (8, 1, 512)]


def _log(rng, lo, hi):
    """A whole number, spread over the logarithm of [lo, hi]."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    while True:
        kind = rng.choice(["decode", "decode", "decode", "flash", "executor", "chunk", "chunk",
                           "chunk", "rope", "gather", "compact"])
        heads, kv_heads, dim = rng.choice(_HEADS)
        kv = rng.choice(["f16", "f16", "q8_0"])
        c = {"kind": kind, **_shape(heads, kv_heads, dim, rng.choice([16, 32, 64]), kv)}
        hi = _log(rng, 48, 16384)
        c["len_max"], c["len_min"] = hi, rng.choice([hi, max(1, hi // rng.randint(2, 8))])
        if kind == "decode":
            c.update(seqs=_log(rng, 1, 64), layers=rng.choice([1, 4, 16]))
        elif kind == "flash":
            c.update(seqs=1, layers=rng.choice([4, 28]), len_max=min(hi, 6000))
            c["len_min"] = c["len_max"]
            c["capacity"] = c["page"] = -(-(c["len_max"] + rng.randint(1, 600)) // 64) * 64
        elif kind == "executor":
            c.update(seqs=_log(rng, 1, 32), layers=rng.choice([4, 16, 28]),
                     tokens=rng.choice([1, 1, 1, 5, 64]), len_max=min(hi, 2500))
            c["len_min"] = min(c["len_min"], c["len_max"])
        elif kind == "chunk":
            c.update(seqs=_log(rng, 1, 8), tokens=_log(rng, 2, 512))
        elif kind == "rope":
            c.update(seqs=_log(rng, 1, 32), tokens=_log(rng, 1, 512), norm=rng.random() < 0.5,
                     v_norm=rng.random() < 0.2, neox=rng.random() < 0.5)
        elif kind == "gather":
            c.update(seqs=_log(rng, 1, 8), layers=rng.choice([1, 4]))
        else:
            c.update(seqs=_log(rng, 1, 8), layers=rng.choice([8, 32]), len_max=min(hi + 500, 4608))
            c["len_min"] = c["len_max"]
        w, rows = work(c), c["seqs"] * c.get("tokens", 1)
        most = 3e10 if kind == "executor" else 1.4e11 if dim > 128 else 2.9e11
        if (0 < w["bytes"] <= 2.2e9 and w["flops"] <= most and _pool_size(c) <= 2.6e9
                # 512-wide heads on a quantized cache attend row by row, over at most
                # 1022 pages: few rows and larger pages are usual there
                and (c["kind"] not in ("chunk", "executor") or dim != 512 or kv == "f16"
                     or (rows <= 64 and max(_held(c)) <= 1000 * c["page"]))):
            return c


# ---- what a pass cannot do without --------------------------------------------

def _lengths(case):
    """Cached tokens of each sequence (the pass's own tokens included for a
    decode, excluded for a chunk), the same for every seed."""
    lo, hi, n = case["len_min"], case["len_max"], case["seqs"]
    r = np.random.default_rng(lo * 7919 + hi)
    return [int(x) for x in r.integers(lo, hi + 1, size=n)]


def _held(case):
    """Tokens that each sequence holds after a pass."""
    more = case["tokens"] if case["kind"] in ("chunk", "executor", "rope") else 0
    return [n + more for n in _lengths(case)]


def _row_bytes(case):
    """One token's K (or V) of one layer in the cache."""
    d = case["kv_heads"] * case["dim"]
    return d * 2 if case["kv"] == "f16" else d + d // 16


def _pages(case):
    if case["kind"] == "flash":  # the whole cache is one page
        return 1
    return sum(-(-n // case["page"]) for n in _held(case)) + 1


def _pool_size(case):
    return case.get("layers", 1) * _pages(case) * case["page"] * _row_bytes(case)


def work(case):
    row, d, kvd = _row_bytes(case), case["dim"], case["kv_heads"] * case["dim"]
    hd = case["heads"] * d
    lens, layers = _lengths(case), case.get("layers", 1)
    tok = case.get("tokens", 1)
    kind = case["kind"]
    if kind in ("decode", "flash"):
        n = sum(lens)
        per = 2 * n * row + len(lens) * (2 * 4 * kvd + 2 * 4 * hd)
        return {"bytes": layers * per, "flops": layers * 4 * hd * n}
    if kind in ("chunk", "executor"):
        new = len(lens) * tok
        pairs = sum(tok * n + tok * (tok + 1) // 2 for n in lens)
        per = 2 * (sum(lens) + new) * row + new * (2 * 4 * kvd + 2 * 4 * hd)
        return {"bytes": layers * per, "flops": layers * 4 * hd * pairs}
    if kind == "rope":
        new = len(lens) * tok
        return {"bytes": new * (2 * 4 * hd + 2 * 4 * kvd + 2 * row), "flops": new * 6 * (hd + kvd)}
    if kind == "gather":  # the output is as long as the longest sequence, zeros past the others
        return {"bytes": layers * 2 * row * (sum(lens) + len(lens) * max(lens)), "flops": 0}
    return {"bytes": 2 * 2 * layers * case["page"] * row * len(_moves(case, 0)), "flops": 0}


# Against 64 bits, attention on f16 caches is 1.1e-4 to 2.1e-4 off (2-norm): the
# fp16 rounding of the probabilities, which another order of the sums or other
# splits draw anew.  On q8_0 caches a chunk is 1e-6 off and a decode over 16k
# tokens 2e-5 (32-bit sums of biased values).  The limits are four times what
# two such results differ by.
def tolerance(case):
    if case["kind"] in ("rope", "gather", "compact"):
        return "exact"  # stored bytes and the rows beside them are defined bit by bit
    return {"rel": 1e-3, "max": 1e-2} if case["kv"] == "f16" else {"rel": 1e-4, "max": 2e-3}


# ---- inputs --------------------------------------------------------------------

def _gen(seed, part):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1000003 + part) & 0x7FFFFFFFFFFF)
    return g


def _randn(gen, *shape):
    return torch.randn(shape, generator=gen, device=DEV, dtype=torch.float32)


def _rows(case, gen, *shape):
    """Rows of K or V: N(0, 1), and 1% outliers where the cache is quantized."""
    x = _randn(gen, *shape)
    if case["kv"] == "q8_0":
        x = torch.where(torch.rand(x.shape, generator=gen, device=DEV) < 0.01, x * 20.0, x)
    return x


def _quantize(x):
    """q8_0 of rows [..., D]: (int8 values [..., D], fp16 scales [..., D / 32])."""
    b = x.view(*x.shape[:-1], -1, 32)
    d = b.abs().amax(-1) / 127.0
    inv = torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
    p = (b * inv.unsqueeze(-1)).double()
    q = (p.sign() * torch.floor(p.abs() + 0.5)).clamp(-127, 127).to(torch.int8)
    return q.view(x.shape), d.half()


def _stored(case, x):
    """The values the cache holds for rows [..., D], as doubles."""
    if case["kv"] == "f16":
        return x.half().double()
    q, d = _quantize(x)
    return (q.view(*d.shape, 32).double() * d.double().unsqueeze(-1)).view(x.shape)


def _pool(case, gen):
    """A filled pool: [layer][page][kv head] regions of page x dim values
    (q8_0: followed by the scales of the region's 32-value blocks)."""
    layers, pages = case.get("layers", 1), _pages(case)
    hk, d, bt = case["kv_heads"], case["dim"], case["page"]
    if case["kv"] == "f16":
        p = torch.empty(layers * pages * hk * bt * d, dtype=torch.float16, device=DEV)
        return p.normal_(generator=gen).view(torch.uint8)
    out = torch.empty((layers * pages, hk, bt * d + bt * d // 16), dtype=torch.uint8, device=DEV)
    step = max(1, (1 << 26) // (hk * bt * d))
    for at in range(0, layers * pages, step):
        n = min(step, layers * pages - at)
        q, s = _quantize(_rows(case, gen, n, hk, bt, d))
        out[at:at + n, :, :bt * d] = q.reshape(n, hk, bt * d).view(torch.uint8)
        out[at:at + n, :, bt * d:] = s.reshape(n, hk, bt * d // 32).view(torch.uint8)
    return out.view(-1)


def _dense(case, pool, layer, pages, n):
    """Tokens [0, n) of a sequence as doubles [n, kv heads, dim]."""
    hk, d, bt = case["kv_heads"], case["dim"], case["page"]
    regions = pool.view(case.get("layers", 1), _pages(case), hk, -1)[layer]
    regions = regions[pages[:-(-n // bt)].long()]
    if case["kv"] == "f16":
        x = regions.view(torch.float16).view(-1, hk, bt, d).double()
    else:
        q = regions[..., :bt * d].contiguous().view(torch.int8).view(-1, hk, bt, d // 32, 32)
        s = regions[..., bt * d:].contiguous().view(torch.float16).view(-1, hk, bt, d // 32, 1)
        x = (q.double() * s.double()).view(-1, hk, bt, d)
    return x.transpose(1, 2).reshape(-1, hk, d)[:n]


def _tables(case, seed):
    """Block tables [seqs, most pages + 1]: a seeded permutation of the pages."""
    need = [-(-n // case["page"]) for n in _held(case)]
    perm = np.random.default_rng(int(seed)).permutation(_pages(case))
    t = np.full((case["seqs"], max(need) + 1), 0xFFFF, dtype=np.uint16)
    at = 0
    for s, n in enumerate(need):
        t[s, :n] = perm[at:at + n]
        at += n
    return torch.from_numpy(t.view(np.int16)).to(DEV)


def _moves(case, seed):
    """(source, destination) of the pages that fill the holes a seeded quarter
    of every sequence's pages leaves at the front of the pool."""
    r = np.random.default_rng(int(seed))
    perm = r.permutation(_pages(case))
    live, at = [], 0
    for n in (-(-x // case["page"]) for x in _held(case)):
        keep = np.sort(r.permutation(n)[:n - n // 4])
        live += [int(x) for x in perm[at:at + n][keep]]
        at += n
    holes = sorted(set(range(len(live))) - set(live))
    return list(zip(sorted(x for x in live if x >= len(live)), holes))


def _geometry(case):
    return emelk.geometry(case.get("layers", 1), case["heads"], case["kv_heads"], case["dim"],
                          case["page"], _pages(case),
                          emelk.KV_F16 if case["kv"] == "f16" else emelk.KV_Q8_0)


def _inputs(case, seed):
    kind, n, d = case["kind"], case["seqs"], case["dim"]
    hd, kvd = case["heads"] * d, case["kv_heads"] * d
    layers, tok = case.get("layers", 1), case.get("tokens", 1)
    i = {"lens": _lengths(case)}
    if kind != "executor":
        i["k_pool"], i["v_pool"] = _pool(case, _gen(seed, 1)), _pool(case, _gen(seed, 2))
    if kind in ("decode", "flash", "executor", "chunk", "rope"):
        i["q"] = _randn(_gen(seed, 3), layers, n, tok, hd)
        i["k"] = _rows(case, _gen(seed, 4), layers, n, tok, kvd)
        i["v"] = _rows(case, _gen(seed, 5), layers, n, tok, kvd)
    if kind == "flash":
        i["tables"] = torch.zeros((1, 1), dtype=torch.int16, device=DEV)
    elif kind not in ("executor", "compact"):
        i["tables"] = _tables(case, seed)
    if kind == "executor" or (kind == "rope" and case["norm"]):
        w = 1.0 + 0.1 * _randn(_gen(seed, 6), 2, d)
        i["q_norm"], i["k_norm"] = w[0], w[1]
    return i


def _history(case, seed, s):
    """The projections of sequence s's cached tokens, of every layer (executor)."""
    kvd, n = case["kv_heads"] * case["dim"], _lengths(case)[s]
    gen = _gen(seed, 100 + s)
    return _rows(case, gen, case["layers"], n, kvd), _rows(case, gen, case["layers"], n, kvd)


# ---- a program's state, and one pass --------------------------------------------

_BASE = 1e6  # RoPE frequency base
_EPS = 1e-6


def prepare(case, seed):
    st = _inputs(case, seed)
    st["case"], st["kind"] = dict(case), case["kind"]
    kind, n, d = case["kind"], case["seqs"], case["dim"]
    layers = case.get("layers", 1)
    scale = st["scale"] = 1.0 / math.sqrt(d)
    lens = st["lens"]
    if kind == "executor":
        _prepare_executor(case, seed, st)
        return st
    g = st["g"] = _geometry(case)
    if kind in ("decode", "flash"):
        for k in ("q", "k", "v"):
            st[k] = st[k].view(layers, n, -1)
        st["out"] = torch.empty_like(st["q"])
        st["kv_lens"] = torch.tensor(lens, dtype=torch.int32, device=DEV)
        st["ws"] = torch.empty(emelk.decode_workspace_bytes(g, n, max(lens)), dtype=torch.uint8,
                               device=DEV)
        most = max(lens)

        def step():
            for l in range(layers):
                if kind == "flash":
                    emelk.decode_contiguous(g, st["k_pool"], st["v_pool"], l, st["q"][l],
                                            st["out"][l], st["kv_lens"], most, case["capacity"],
                                            scale, st["ws"], k_rows=st["k"][l], v_rows=st["v"][l])
                else:
                    emelk.decode_append(g, st["k_pool"], st["v_pool"], l, st["k"][l], st["v"][l],
                                        st["q"][l], st["out"][l], st["kv_lens"], most,
                                        st["tables"], scale, st["ws"])

        st["step"] = step
        if layers > 1:  # a serving loop's step: captured once, replayed per token
            step()
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                step()
            st["graph"] = graph
            st["step"] = graph.replay
    elif kind == "chunk":
        for k in ("q", "k", "v"):
            st[k] = st[k][0]
        st["out"] = torch.empty_like(st["q"])
        st["start"] = torch.tensor(lens, dtype=torch.int32, device=DEV)
    elif kind == "rope":
        for k in ("q", "k", "v"):
            st[k] = st[k][0]
        st["out"] = torch.empty_like(st["q"])
        st["start"] = torch.tensor(lens, dtype=torch.int32, device=DEV)
        st["rope"] = emelk.RopeTable(d, d, max(_held(case)), _BASE, _pairing(case))
    elif kind == "gather":
        row = case["dim"] * 2 if case["kv"] == "f16" else case["dim"] // 32 * 34
        shape = (layers, n, case["kv_heads"], max(lens), row)
        st["k_out"] = torch.empty(shape, dtype=torch.uint8, device=DEV)
        st["v_out"] = torch.empty_like(st["k_out"])
        st["lengths"] = torch.tensor(lens, dtype=torch.int32, device=DEV)
    else:
        moves = np.array(_moves(case, seed), dtype=np.int32).reshape(-1, 2)
        st["moves"] = torch.tensor(moves, dtype=torch.int32, device=DEV)
    return st


def _pairing(case):
    return emelk.NEOX_PAIRING if case.get("neox", True) else emelk.NORMAL_PAIRING


def _prepare_executor(case, seed, st):
    n, layers, page, tok = case["seqs"], case["layers"], case["page"], case["tokens"]
    g = _geometry(case)
    actor = emelk.KvActor()
    ok, err = actor.reserve(n, _pages(case), page)
    assert ok, err
    actor.set_free_order(np.random.default_rng(int(seed)).permutation(_pages(case)).astype(np.uint16))
    cache = emelk.KvCache(g)
    most = max(_held(case))
    rope = emelk.RopeTable(case["dim"], case["dim"], most, _BASE, _pairing(case))
    dec = emelk.BatchDecoder(g, actor, cache, rope, max_batch=n, max_kv_len=most)
    st.update(actor=actor, cache=cache, rope=rope, dec=dec, ids=list(range(n)))
    for s, length in enumerate(st["lens"]):
        assert actor.allocate_sequence(s)[0]
        k, v = _history(case, seed, s)
        q = _randn(_gen(seed, 7), length, case["heads"] * case["dim"])
        out = torch.empty_like(q)
        dec.begin_step([s], length)
        for l in range(layers):
            dec.layer(l, q, torch.empty_like(q), k[l], v[l], out, st["scale"], st["q_norm"],
                      st["k_norm"], False, _EPS)
    st["q_roped"] = torch.empty_like(st["q"])
    st["out"] = torch.empty_like(st["q"])


def run(st):
    kind = st["kind"]
    if kind in ("decode", "flash"):
        st["step"]()
        return st["out"]
    if kind == "executor":
        case, dec = st["case"], st["dec"]
        dec.begin_step(st["ids"], case["tokens"])
        for l in range(case["layers"]):
            dec.layer(l, st["q"][l], st["q_roped"][l], st["k"][l], st["v"][l], st["out"][l],
                      st["scale"], st["q_norm"], st["k_norm"], False, _EPS)
        for s in st["ids"]:
            st["actor"].rollback_slots(s, case["tokens"])
        return st["out"], st["q_roped"]
    if kind == "chunk":
        emelk.append(st["g"], st["k_pool"], st["v_pool"], 0, st["k"], st["v"], st["start"],
                     st["tables"])
        emelk.prefill_chunk(st["g"], st["k_pool"], st["v_pool"], 0, st["q"], st["out"],
                            st["start"], st["tables"], st["scale"])
        return st["out"], _whole(st)
    if kind == "rope":
        emelk.qkv_rope_append(st["g"], st["k_pool"], st["v_pool"], 0, st["q"], st["out"], st["k"],
                              st["v"], st["start"], st["tables"], st["rope"], st.get("q_norm"),
                              st.get("k_norm"), st["case"]["v_norm"], _EPS)
        return st["out"], _whole(st)
    if kind == "gather":
        for l in range(st["case"]["layers"]):
            emelk.gather(st["g"], st["k_pool"], st["v_pool"], l, st["lengths"], st["tables"],
                         st["k_out"][l], st["v_out"][l], int(st["k_out"].shape[3]))
        return st["k_out"], st["v_out"]
    emelk.copy_blocks(st["g"], st["k_pool"], st["v_pool"], st["moves"])
    return _whole(st)


def _whole(st):
    """Both pools, as words."""
    return [st["k_pool"].view(torch.int32), st["v_pool"].view(torch.int32)]


# ---- 64-bit results ------------------------------------------------------------

def _attend(case, q, k, v, first):
    """Causal attention in doubles: q [rows, heads * dim] at positions first,
    first + 1, ...; k, v [tokens, kv heads, dim].  q is fp16, as the cache's
    attention defines it."""
    h, hk, d = case["heads"], case["kv_heads"], case["dim"]
    rows, group = q.shape[0], h // hk
    out = torch.empty((rows, h, d), dtype=torch.float64, device=DEV)
    qd = q.half().double().view(rows, h, d)
    pos = torch.arange(first, first + rows, device=DEV).view(-1, 1)
    ok = torch.arange(k.shape[0], device=DEV).view(1, -1) <= pos
    for j in range(hk):  # the rows of one KV head's query heads together
        heads = slice(j * group, (j + 1) * group)
        s = torch.matmul(qd[:, heads].reshape(-1, d), k[:, j].t().contiguous()) / math.sqrt(d)
        s = s.view(rows, group, -1).masked_fill(~ok.unsqueeze(1), -math.inf)
        o = torch.matmul(torch.softmax(s, -1).view(rows * group, -1), v[:, j].contiguous())
        out[:, heads] = o.view(rows, group, d)
    return out.view(rows, h * d)


def _turned(case, x, weight, first):
    """Head norm (weight or None) and RoPE of rows [tokens, heads * dim] at
    positions first, first + 1, ..., in doubles.  The angles are the 32-bit
    ones that the recurrence over the pairs gives."""
    d, n = case["dim"], x.shape[0]
    y = x.double().view(n, -1, d)
    if weight is not None:
        y = y / torch.sqrt((y * y).mean(-1, keepdim=True) + _EPS) * weight.double()
    theta = np.arange(first, first + n, dtype=np.float32)
    step = np.float32(np.power(np.float32(_BASE), np.float32(-2.0 / d)))
    angles = np.empty((n, d // 2), dtype=np.float32)
    for p in range(d // 2):
        angles[:, p] = theta
        theta = theta * step
    a = torch.from_numpy(angles).to(DEV).double().unsqueeze(1)
    c, s = torch.cos(a), torch.sin(a)
    if case.get("neox", True):
        x0, x1 = y[..., :d // 2], y[..., d // 2:]
        y = torch.cat([x0 * c - x1 * s, x0 * s + x1 * c], -1)
    else:
        x0, x1 = y[..., 0::2], y[..., 1::2]
        y = torch.stack([x0 * c - x1 * s, x0 * s + x1 * c], -1)
    return y.reshape(n, -1)


def exact(case, seed):
    kind, hk, d = case["kind"], case["kv_heads"], case["dim"]
    if kind in ("gather", "compact"):
        return None
    i = _inputs(case, seed)
    lens, layers, tok = i["lens"], case.get("layers", 1), case.get("tokens", 1)
    if kind in ("decode", "flash"):
        out = torch.empty((layers, case["seqs"], case["heads"] * d), dtype=torch.float64, device=DEV)
        for l in range(layers):
            for s, n in enumerate(lens):
                kv = []
                for pool, new in ((i["k_pool"], i["k"]), (i["v_pool"], i["v"])):
                    old = _dense(case, pool, l, i["tables"][s].to(torch.int32) & 0xFFFF, n - 1)
                    kv.append(torch.cat([old, _stored(case, new[l, s].view(1, hk, d))]))
                out[l, s] = _attend(case, i["q"][l, s], *kv, n - 1)[0]
        return out
    if kind == "chunk":
        out = torch.empty((case["seqs"], tok, case["heads"] * d), dtype=torch.float64, device=DEV)
        for s, n in enumerate(lens):
            kv = []
            for pool, new in ((i["k_pool"], i["k"]), (i["v_pool"], i["v"])):
                old = _dense(case, pool, 0, i["tables"][s].to(torch.int32) & 0xFFFF, n)
                kv.append(torch.cat([old, _stored(case, new[0, s].view(tok, hk, d))]))
            out[s] = _attend(case, i["q"][0, s], *kv, n)
        return out, [None, None]
    if kind == "rope":
        out = torch.stack([_turned(case, i["q"][0, s], i.get("q_norm"), n)
                           for s, n in enumerate(lens)])
        return out, [None, None]
    out = torch.empty((layers, case["seqs"], tok, case["heads"] * d), dtype=torch.float64,
                      device=DEV)
    roped = torch.empty_like(out)
    for s, n in enumerate(lens):
        hist = _history(case, seed, s)
        for l in range(layers):
            rows = [torch.cat([hist[0][l], i["k"][l, s]]), torch.cat([hist[1][l], i["v"][l, s]])]
            k = _stored(case, _turned(case, rows[0], i["k_norm"], 0).float().view(-1, hk, d))
            v = _stored(case, rows[1].view(-1, hk, d))
            roped[l, s] = _turned(case, i["q"][l, s], i["q_norm"], n)
            out[l, s] = _attend(case, roped[l, s].float(), k, v, n)
    return out, roped
