"""Measured workloads of the quantized KV-cache path.

Each case is one pass through the public entry points: a decode step over a few
attention layers, a batched decode, a suffix (prompt, chat turn, verification) over a
cached prefix, a bulk store of prompt rows, or a fork of one session into many.
``listed()`` gives fixed cases, ``draw(rng)`` further ones of the same ranges;
``prepare`` makes what a serving program holds before the call (filled caches, block
tables, workspaces, output buffers, for a decode loop its captured graph), ``run`` is
the pass, ``work`` the bytes and operations it cannot do without, ``exact`` the same
results in 64-bit torch from the inputs alone.
"""
from __future__ import annotations

import math

import torch

import miinfer_amd as m
from miinfer_amd import _lib
from miinfer_amd import reuse as mreuse

BLOCK = 32  # values per q8_0 block
THETA, EPSILON = 1.0e7, 1.0e-6
DEV = "cuda"


# ---- the cases --------------------------------------------------------------------

def listed():
    gqa128 = {"q_heads": 32, "kv_heads": 8, "head_dim": 128}  # Qwen3-8B-shaped layer
    gqa256 = {"q_heads": 24, "kv_heads": 4, "head_dim": 256}  # the larger-head layer
    return [
        # first tokens of a session: one layer, called directly; launches and latency
        {"name": "decode_257", "kind": "decode", **gqa128, "mode": "q8", "q": "f16", "context": 257,
         "max_context": 512, "layers": 1, "graph": False, "rows": "f16", "gate": False},
        # the headline step: append and attend at 32k, a decode graph over 8 layers
        {"name": "decode_32k", "kind": "decode", **gqa128, "mode": "q8", "q": "f16", "context": 32768,
         "max_context": 32768, "layers": 8, "graph": True, "rows": "f16", "gate": False},
        # a decode graph captured once for a 16k session, at an odd position inside it:
        # fp32 rows with the K norm and rotation, fp32 query, gated output
        {"name": "decode_gated_9k", "kind": "decode", **gqa256, "mode": "q8", "q": "f32", "context": 9001,
         "max_context": 16384, "layers": 8, "graph": True, "rows": "f32", "gate": True},
        # the fp16 cache (the unquantized mode): store, then attend
        {"name": "decode_fp16_16k", "kind": "decode", **gqa256, "mode": "f16", "q": "f16", "context": 16384,
         "max_context": 16384, "layers": 8, "graph": True, "rows": "f16", "gate": False},
        # batched paged decode over long, ragged contexts
        {"name": "batch_long_16", "kind": "batch", **gqa256, "q": "f16", "batch": 16, "low": 1024, "high": 65536,
         "gate": False},
        # a serving batch of ordinary chats
        {"name": "batch_chat_48", "kind": "batch", **gqa128, "q": "f16", "batch": 48, "low": 64, "high": 4096,
         "gate": False},
        # verification of a few drafted tokens over a cached context
        {"name": "suffix_verify_5", "kind": "suffix", **gqa256, "q": "f16", "prefix": 8187, "tokens": 5,
         "paged": False, "gate": False, "exact": False, "layers": 4, "graph": True},
        # a chat turn over the cached conversation, paged, fp32 query, gated output
        {"name": "suffix_turn_77", "kind": "suffix", **gqa256, "q": "f32", "prefix": 3001, "tokens": 77,
         "paged": True, "gate": True, "exact": False, "layers": 4, "graph": True},
        # a 512-token chunk over an 8k prefix
        {"name": "suffix_512_8k", "kind": "suffix", **gqa256, "q": "f16", "prefix": 8192, "tokens": 512,
         "paged": False, "gate": False, "exact": False, "layers": 1, "graph": False},
        # a whole prompt into an empty cache
        {"name": "prefill_2048", "kind": "suffix", **gqa128, "q": "f16", "prefix": 0, "tokens": 2048,
         "paged": False, "gate": False, "exact": False, "layers": 1, "graph": False},
        # store of a prompt's rows with the K norm and rotation, at an odd position
        {"name": "append_8195", "kind": "append", **gqa256, "rows": "f32", "base": 77, "tokens": 8195},
        # one prefix forked into 24 sessions: block tables, partial pages, recurrent state
        {"name": "fork_24", "kind": "fork", "kv_heads": 4, "head_dim": 256, "prefix": 8300, "forks": 24,
         "attn_layers": 8, "gdn_layers": 24},
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    shape = rng.choice([(32, 8, 128), (24, 4, 256)])
    c = {"q_heads": shape[0], "kv_heads": shape[1], "head_dim": shape[2]}
    kind = rng.choice(["decode", "decode", "batch", "batch", "suffix", "suffix", "suffix", "append", "fork"])
    if kind == "decode":
        mode = rng.choice(["q8", "q8", "q8", "f16"])
        context = _log(rng, 16, 32768 if mode == "q8" else 16384)
        top = max(512, 1 << (context - 1).bit_length())  # the session's capacity
        return {"kind": kind, **c, "mode": mode, "q": rng.choice(["f16", "f32"]), "context": context,
                "max_context": rng.choice([top, -(-context // 64) * 64]), "layers": rng.randint(2, 8),
                "graph": True, "rows": rng.choice(["f16", "f32"]) if mode == "q8" else "f16",
                "gate": rng.random() < 0.5}
    if kind == "batch":
        high = _log(rng, 512, 32768)
        return {"kind": kind, **c, "q": rng.choice(["f16", "f32"]), "batch": rng.randint(2, max(4, min(96, 400000 // high))),
                "low": max(1, high // rng.choice([2, 8, 64])), "high": high, "gate": rng.random() < 0.5}
    if kind == "suffix":
        tokens = _log(rng, 2, 2048)
        exact = rng.random() < 0.2
        # no more pairs than the 512-token chunk over 8k has
        most = (1.8e6 if exact else 4.2e6) / tokens - tokens / 2
        prefix = rng.choice([0, _log(rng, 64, min(16384, most))]) if most > 64 else 0
        small = tokens <= 128
        return {"kind": kind, **c, "q": rng.choice(["f16", "f32"]), "prefix": prefix, "tokens": tokens,
                "paged": rng.random() < 0.5, "gate": rng.random() < 0.5, "exact": exact,
                "layers": 4 if small else 1, "graph": small}
    if kind == "append":
        return {"kind": kind, **c, "rows": rng.choice(["f16", "f32"]), "base": rng.randint(0, 300),
                "tokens": _log(rng, 64, 8192)}
    return {"kind": kind, "kv_heads": shape[1], "head_dim": shape[2], "prefix": _log(rng, 300, 8300),
            "forks": rng.randint(2, 24), "attn_layers": rng.randint(2, 8), "gdn_layers": rng.randint(4, 24)}


# ---- inputs -----------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _randn(g, shape, dtype):
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32).to(dtype)


def _dtype(name):
    return torch.float16 if name == "f16" else torch.float32


def _up(n, unit):
    return -(-n // unit) * unit


def _lengths(case):
    """Context lengths of a batch, spread evenly over [low, high] in a mixed order."""
    n, lo, hi = case["batch"], case["low"], case["high"]
    return [lo + int((hi - lo) * ((0.5 + i * 0.6180339887) % 1.0)) for i in range(n)]


def _inputs(case, seed):
    """Every random tensor of a case, from the seed alone."""
    g = _gen(seed)
    kind = case["kind"]
    if kind == "fork":
        return g
    hq, hk, d = case["q_heads"], case["kv_heads"], case["head_dim"]
    x = {}
    if kind == "decode":
        n = case["layers"]
        rows = _dtype(case["rows"])
        x["k"] = [_randn(g, (case["context"] - 1, hk, d), torch.float16) for _ in range(n)]
        x["v"] = [_randn(g, (case["context"] - 1, hk, d), torch.float16) for _ in range(n)]
        x["q"] = [_randn(g, (1, hq, d), _dtype(case["q"])) for _ in range(n)]
        x["k_new"] = [_randn(g, (1, hk, d), rows) for _ in range(n)]
        x["v_new"] = [_randn(g, (1, hk, d), rows) for _ in range(n)]
        if case["rows"] == "f32":
            x["norm"] = [0.5 + torch.rand((d,), generator=g, device=DEV) for _ in range(n)]
        if case["gate"]:
            x["gate"] = [_randn(g, (1, hq, d), torch.float32) for _ in range(n)]
    elif kind == "batch":
        b = case["batch"]
        x["k"] = [_randn(g, (L - 1, hk, d), torch.float16) for L in _lengths(case)]
        x["v"] = [_randn(g, (L - 1, hk, d), torch.float16) for L in _lengths(case)]
        x["q"] = _randn(g, (b, hq, d), _dtype(case["q"]))
        x["k_new"] = _randn(g, (b, hk, d), torch.float16)
        x["v_new"] = _randn(g, (b, hk, d), torch.float16)
        if case["gate"]:
            x["gate"] = _randn(g, (b, hq, d), torch.float32)
    elif kind == "suffix":
        n, p, t = case["layers"], case["prefix"], case["tokens"]
        x["k"] = [_randn(g, (p, hk, d), torch.float16) for _ in range(n)]
        x["v"] = [_randn(g, (p, hk, d), torch.float16) for _ in range(n)]
        x["q"] = [_randn(g, (t, hq, d), _dtype(case["q"])) for _ in range(n)]
        x["k_new"] = [_randn(g, (t, hk, d), torch.float16) for _ in range(n)]
        x["v_new"] = [_randn(g, (t, hk, d), torch.float16) for _ in range(n)]
        if case["gate"]:
            x["gate"] = [_randn(g, (t, hq, d), torch.float32) for _ in range(n)]
    else:
        t = case["tokens"]
        x["k"] = _randn(g, (t, hk, d), _dtype(case["rows"]))
        x["v"] = _randn(g, (t, hk, d), _dtype(case["rows"]))
        if case["rows"] == "f32":
            x["norm"] = 0.5 + torch.rand((d,), generator=g, device=DEV)
    x["g"] = g
    return x


def _planes(cache):
    return [p for p in (cache.k_codes, cache.k_scales, cache.v_codes, cache.v_scales) if p is not None]


def _paged(hk, d, rows, width, page, g):
    """A paged cache whose sequences (page counts `rows`) own random physical pages; block
    tables of `width` entries."""
    total = sum(rows)
    perm = torch.randperm(total, generator=g, device=DEV).to(torch.int32)
    table = torch.full((len(rows), width), -1, dtype=torch.int32, device=DEV)
    at = 0
    for b, n in enumerate(rows):
        table[b, :n] = perm[at:at + n]
        at += n
    return m.KvCache.paged_cache(hk, d, total, table, page_tokens=page)


# ---- prepare / run ----------------------------------------------------------------

def _ptr(t):
    return None if t is None else t.data_ptr()


def _decode_layer(s, i):
    """One layer's step of a decode loop: store the new row, attend."""
    c = s["case"]
    x = s["x"]
    gate = x["gate"][i] if c["gate"] else None
    out = None if c["gate"] else s["out"][i]
    gated = s["out"][i] if c["gate"] else None
    cache, ws = s["caches"][i], s["ws"]
    if c["rows"] == "f32":
        # the fused step with the K norm and rotation exists in the C interface only
        _lib.call("miikv_decode_append_attn_f32", cache.view, _ptr(x["k_new"][i]), _ptr(x["v_new"][i]),
               _ptr(x["norm"][i]), THETA, EPSILON, _ptr(x["q"][i]), 0 if c["q"] == "f16" else 1, c["q_heads"],
               1.0 / math.sqrt(c["head_dim"]), 1, None, _ptr(s["state"]), c["max_context"], _ptr(out),
               _ptr(gate), _ptr(gated), None, _ptr(ws.buf), ws.bytes, torch.cuda.current_stream().cuda_stream)
        return
    k_new, v_new = x["k_new"][i], x["v_new"][i]
    if c["mode"] == "f16":  # fp16 planes: the row is stored first
        cache.append(k_new, v_new, decode_state=s["state"])
        k_new = v_new = None
    m.decode_attention(cache, x["q"][i], decode_state=s["state"], max_context=c["max_context"], gate=gate, out=out,
                       gated_out=gated, k_new=k_new, v_new=v_new, workspace=ws)


def _suffix_layer(s, i):
    c = s["case"]
    x = s["x"]
    gate = x["gate"][i] if c["gate"] else None
    m.suffix_attention(s["caches"][i], x["q"][i], c["prefix"], gate=gate,
                       out=None if c["gate"] else s["out"][i], gated_out=s["out"][i] if c["gate"] else None,
                       k_new=x["k_new"][i], v_new=x["v_new"][i], workspace=s["ws"], exact=c["exact"])


def _capture(s, layer, layers):
    """The layers' launches as one graph, as a serving loop captures its step."""
    layer(s, 0)  # loads the kernels
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for i in range(layers):
            layer(s, i)
    return graph


def prepare(case, seed):
    kind = case["kind"]
    x = _inputs(case, seed)
    s = {"case": case, "x": x}
    hk, d = case["kv_heads"], case["head_dim"]
    if kind == "decode":
        n, hq = case["layers"], case["q_heads"]
        quant = _lib.KV_Q8_Q8 if case["mode"] == "q8" else _lib.KV_FP16_FP16
        s["caches"] = [m.KvCache.contiguous(hk, d, case["max_context"], quant_mode=quant) for _ in range(n)]
        for c, k, v in zip(s["caches"], x.pop("k"), x.pop("v")):
            if k.shape[0]:
                c.append(k, v)
        s["state"] = m.make_decode_state(case["context"] - 1)
        s["ws"] = m.DecodeWorkspace(s["caches"][0], hq, 1, case["max_context"])
        s["out"] = [torch.empty((1, hq, d), dtype=torch.float32, device=DEV) for _ in range(n)]
        s["graph"] = _capture(s, _decode_layer, n) if case["graph"] else None
    elif kind == "batch":
        lens, page = _lengths(case), 256
        s["cache"] = _paged(hk, d, [_up(L, page) // page for L in lens], _up(case["high"], page) // page, page, x["g"])
        for b, (k, v) in enumerate(zip(x.pop("k"), x.pop("v"))):
            if k.shape[0]:
                s["cache"].append(k, v, seq=b)
        s["lengths"] = torch.tensor(lens, dtype=torch.int32, device=DEV)
        s["max_context"] = _up(case["high"], page)
        s["ws"] = m.DecodeWorkspace(s["cache"], case["q_heads"], case["batch"], s["max_context"])
        s["out"] = torch.empty((case["batch"], case["q_heads"], d), dtype=torch.float32, device=DEV)
    elif kind == "suffix":
        n, hq, p, t = case["layers"], case["q_heads"], case["prefix"], case["tokens"]
        s["caches"] = []
        for k, v in zip(x.pop("k"), x.pop("v")):
            if case["paged"]:
                pages = _up(p + t, 256) // 256
                c = _paged(hk, d, [pages], pages, 256, x["g"])
            else:
                c = m.KvCache.contiguous(hk, d, _up(p + t, 64))
            if p:
                c.append(k, v)
            s["caches"].append(c)
        need = m.suffix_workspace_bytes(s["caches"][0], hq, t, exact=case["exact"])
        s["ws"] = torch.empty(need, dtype=torch.uint8, device=DEV)
        s["out"] = [torch.empty((t, hq, d), dtype=torch.float32, device=DEV) for _ in range(n)]
        s["graph"] = _capture(s, _suffix_layer, n) if case["graph"] else None
    elif kind == "append":
        s["cache"] = m.KvCache.contiguous(hk, d, _up(case["base"] + case["tokens"], 64))
    else:
        page, p, n = 256, case["prefix"], case["forks"]
        pages = _up(p, page) // page
        s["pool"] = mreuse.PagePool(pages + n)
        row = [s["pool"].alloc() for _ in range(pages)]
        s["row"] = torch.tensor(row, dtype=torch.int32).numpy()
        table = torch.tensor([row], dtype=torch.int32, device=DEV)
        s["caches"] = []
        for _ in range(case["attn_layers"]):
            c = m.KvCache.paged_cache(hk, d, pages + n, table, page_tokens=page)
            c.append(_randn(x, (p, hk, d), torch.float16), _randn(x, (p, hk, d), torch.float16))
            s["caches"].append(c)
        make = lambda: mreuse.RecurrentStates(case["gdn_layers"], 16 * 128 * 128, 8192 * 3)  # noqa: E731
        s["src"] = make()
        s["src"].buf.normal_(generator=x)
        s["dst"] = [make() for _ in range(n)]
        s["live"] = None
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "decode":
        if s["graph"] is not None:
            s["graph"].replay()
        else:
            for i in range(case["layers"]):
                _decode_layer(s, i)
        return s["out"], [_planes(c) for c in s["caches"]]
    if kind == "batch":
        x = s["x"]
        gate = x["gate"] if case["gate"] else None
        m.decode_attention(s["cache"], x["q"], lengths=s["lengths"], max_context=s["max_context"], gate=gate,
                           out=None if case["gate"] else s["out"], gated_out=s["out"] if case["gate"] else None,
                           k_new=x["k_new"], v_new=x["v_new"], workspace=s["ws"])
        return s["out"], _planes(s["cache"])
    if kind == "suffix":
        if s["graph"] is not None:
            s["graph"].replay()
        else:
            for i in range(case["layers"]):
                _suffix_layer(s, i)
        return s["out"], [_planes(c) for c in s["caches"]]
    if kind == "append":
        x = s["x"]
        if case["rows"] == "f32":
            s["cache"].append_f32(x["k"], x["v"], case["base"], k_norm_weight=x["norm"], theta=THETA, epsilon=EPSILON)
        else:
            s["cache"].append(x["k"], x["v"], case["base"])
        return _planes(s["cache"])
    if s["live"] is not None:  # the previous pass's sessions end
        for r in s["live"]:
            s["pool"].release(r, case["prefix"], 256)
    s["live"], copies = s["pool"].fork_many(s["row"], case["prefix"], 256, case["forks"])
    for c in s["caches"]:
        mreuse.run_page_copies(c, copies)
    mreuse.clone_states(s["src"], s["dst"])
    return [_planes(c) for c in s["caches"]], [r.buf for r in s["dst"]]


# ---- what a pass cannot do without --------------------------------------------------

def _kv_bytes(case, tokens, mode="q8"):
    per = case["head_dim"] * 2 if mode == "f16" else case["head_dim"] + case["head_dim"] // 16
    return tokens * 2 * case["kv_heads"] * per


def work(case):
    kind = case["kind"]
    if kind == "fork":
        partial = case["prefix"] % 256 != 0
        page = 2 * 256 * case["kv_heads"] * (case["head_dim"] + case["head_dim"] // 16)
        state = case["gdn_layers"] * (16 * 128 * 128 + 8192 * 3) * 4
        return {"bytes": (case["attn_layers"] * page * (1 + case["forks"]) if partial else 0) + state * (1 + case["forks"]),
                "flops": 0}
    hq, hk, d = case["q_heads"], case["kv_heads"], case["head_dim"]
    if kind == "append":
        row = 2 * hk * d * (4 if case["rows"] == "f32" else 2)
        return {"bytes": case["tokens"] * row + _kv_bytes(case, case["tokens"]), "flops": 0}
    qsize = 2 if case["q"] == "f16" else 4
    if kind == "decode":
        new = 2 * hk * d * (4 if case["rows"] == "f32" else 2)
        io = hq * d * (qsize + 4 + (4 if case["gate"] else 0)) + new
        return {"bytes": case["layers"] * (_kv_bytes(case, case["context"], case["mode"]) + io),
                "flops": case["layers"] * 4 * hq * d * case["context"]}
    if kind == "batch":
        tokens = sum(_lengths(case))
        io = hq * d * (qsize + 4 + (4 if case["gate"] else 0)) + 2 * hk * d * 2
        return {"bytes": _kv_bytes(case, tokens) + case["batch"] * io, "flops": 4 * hq * d * tokens}
    p, t = case["prefix"], case["tokens"]
    io = t * (hq * d * (qsize + 4 + (4 if case["gate"] else 0)) + 2 * hk * d * 2)
    return {"bytes": case["layers"] * (_kv_bytes(case, p + t) + io),
            "flops": case["layers"] * 4 * hq * d * (t * p + t * (t + 1) // 2)}


# Stored codes, scales and copies are bytes.  Attention over fp16 operands: about four
# times its distance from the 64-bit result (2.7e-4 for a decode, whose products are
# exact and probabilities rounded to fp16 once; 4.7e-4 for a suffix, which rounds query
# and keys as well).
def tolerance(case):
    if case["kind"] in ("append", "fork"):
        return "exact"
    return {"rel": 2e-3 if case["kind"] == "suffix" else 1.2e-3}


# ---- the same in 64 bits ------------------------------------------------------------

def _stored(x, mode):
    """Rows [n, heads, D] as the cache holds them, in 64 bits."""
    if mode == "f16":
        return x.to(torch.float16).double()
    b = x.float().reshape(*x.shape[:-1], x.shape[-1] // BLOCK, BLOCK)
    top = b.abs().amax(-1, keepdim=True)
    scale = torch.where(top > 0, top / 127.0, torch.ones_like(top))
    code = torch.clamp(torch.round(b * (1.0 / scale)), -128, 127)
    return (code.double() * scale.to(torch.float16).double()).reshape(x.shape)


def _norm_rope(x, w, pos):
    y = x.double()
    y = y / torch.sqrt((y * y).mean(-1, keepdim=True) + EPSILON) * w.double()
    ang = pos * THETA ** (-2.0 * torch.arange(32, device=DEV, dtype=torch.float64) / 64.0)
    a, b = y[..., :32].clone(), y[..., 32:64].clone()
    y[..., :32] = a * torch.cos(ang) - b * torch.sin(ang)
    y[..., 32:64] = a * torch.sin(ang) + b * torch.cos(ang)
    return y


def _attend(q, k, v, base, gate):
    """q [t, hq, D] at positions base.. over k, v [n, hk, D] (64 bits), causal."""
    t, hq, d = q.shape
    g = hq // k.shape[1]
    out = torch.empty((t, hq, d), dtype=torch.float64, device=DEV)
    hidden = torch.arange(k.shape[0], device=DEV)[None, :] > base + torch.arange(t, device=DEV)[:, None]
    for h in range(hq):
        s = (q[:, h].double() @ k[:, h // g].T.contiguous()) / math.sqrt(d)
        out[:, h] = torch.softmax(s.masked_fill(hidden, -math.inf), -1) @ v[:, h // g]
    return out * torch.sigmoid(gate.double()) if gate is not None else out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("append", "fork"):
        return None
    x = _inputs(case, seed)
    if kind == "decode":
        outs = []
        for i in range(case["layers"]):
            k_new = x["k_new"][i]
            if case["rows"] == "f32":
                k_new = _norm_rope(k_new, x["norm"][i], case["context"] - 1)
            k = _stored(torch.cat([x["k"][i].float(), k_new.float()]), case["mode"])
            v = _stored(torch.cat([x["v"][i].float(), x["v_new"][i].float()]), case["mode"])
            outs.append(_attend(x["q"][i], k, v, case["context"] - 1, x["gate"][i] if case["gate"] else None))
        return outs, None
    if kind == "batch":
        outs = []
        for b in range(case["batch"]):
            k = _stored(torch.cat([x["k"][b], x["k_new"][b:b + 1]]), "q8")
            v = _stored(torch.cat([x["v"][b], x["v_new"][b:b + 1]]), "q8")
            outs.append(_attend(x["q"][b:b + 1], k, v, k.shape[0] - 1, x["gate"][b:b + 1] if case["gate"] else None))
        return torch.cat(outs), None
    outs = []
    for i in range(case["layers"]):
        k = _stored(torch.cat([x["k"][i], x["k_new"][i]]), "q8")
        v = _stored(torch.cat([x["v"][i], x["v_new"][i]]), "q8")
        outs.append(_attend(x["q"][i], k, v, case["prefix"], x["gate"][i] if case["gate"] else None))
    return outs, None
