"""The work a program has this package do, as timed cases.

The shapes are the model's attention (32 query heads over 4 kv heads of 128,
hidden 2048, 128 experts), at the lengths its serving loop meets: one token at
a short, an ordinary and a long context, a prompt's first chunk, a chunk after
a reused prefix, a few rows of a follow-up turn, a long prompt's later chunk,
and the router for a token and for a chunk.

A case is a dict of plain values; its ``kind`` picks the entry points:

- ``decode``: decode_attention for every layer of a token, captured once and
  replayed (the way the serving loop runs its per-token layer sequence);
- ``step``: decode_step called eagerly (norm, RoPE, append, attention);
- ``token``: attn_block_decode_dev for every layer of a token, one graph with
  the position in device memory;
- ``prefill``: prefill_chunk of one layer in one of its three modes;
- ``block``: attn_block_prefill, a layer's whole attention half for a chunk;
- ``router``: router_topk.

Calls that append start by truncating the cache to the case's prefix, as a
program does that reuses one, so a pass can be repeated on its state.
"""
from __future__ import annotations

import math

import torch

import ramvamp_amd as rv
from ramvamp_amd import block as B
from ramvamp_amd import projections as P
from ramvamp_amd import router as R

HEADS, KV_HEADS, DIM, HIDDEN = 32, 4, 128, 2048
Q_DIM, KV_DIM = HEADS * DIM, KV_HEADS * DIM
GROUP = HEADS // KV_HEADS
EPS, THETA, SCALE = 1e-6, 1e6, DIM ** -0.5
FORMATS = {"q4": P.Q4_K, "q5": P.Q5_K, "q6": P.Q6_K, "q8": P.Q8_0}
BLOCK = {"q4": (256, 144), "q5": (256, 176), "q6": (256, 210), "q8": (32, 34)}  # weights, bytes


def listed():
    return [
        # A token early in a conversation: every launch is short, so their number and their gaps count.
        {"name": "decode_48x100_f16", "kind": "decode", "layers": 48, "ctx": 100, "elem": "f16"},
        # The headline: 48 layers over 4096 cached positions of an fp32 cache.
        {"name": "decode_48x4096_f32", "kind": "decode", "layers": 48, "ctx": 4096, "elem": "f32"},
        # A token at the end of a long document, in the model's cache format.
        {"name": "decode_4x32768_f16", "kind": "decode", "layers": 4, "ctx": 32768, "elem": "f16"},
        # One eager step of a program that drives the cache itself, a call per token.
        {"name": "step_512_f32", "kind": "step", "ctx": 512, "elem": "f32"},
        # A token through the attention blocks of 16 layers, at an odd position.
        {"name": "token_16x2003_f16", "kind": "token", "layers": 16, "ctx": 2003, "elem": "f16", "q": "q4", "v": "q6",
         "o": "q5"},
        # A prompt's first chunk: nothing cached, the causal triangle alone.
        {"name": "prefill_512_at_0_f16", "kind": "prefill", "mode": "f16", "rows": 512, "start": 0, "elem": "f16"},
        # A chunk behind a reused prefix at full precision.
        {"name": "prefill_512_at_3449_exact", "kind": "prefill", "mode": "exact", "rows": 512, "start": 3449,
         "elem": "f32"},
        # A late chunk of a long prompt: the largest products.
        {"name": "prefill_1024_at_12000_bf16", "kind": "prefill", "mode": "bf16", "rows": 1024, "start": 12000,
         "elem": "f16"},
        # A layer's attention half for a chunk behind a reused prefix.
        {"name": "block_512_at_3449_f16", "kind": "block", "mode": "f16", "rows": 512, "start": 3449, "elem": "f16",
         "q": "q4", "v": "q6", "o": "q5"},
        # A follow-up turn of a chat: a ragged few rows behind what is cached.
        {"name": "block_77_at_901_exact", "kind": "block", "mode": "exact", "rows": 77, "start": 901, "elem": "f16",
         "q": "q5", "v": "q4", "o": "q6"},
        # The experts of one token, and of a chunk.
        {"name": "router_1", "kind": "router", "rows": 1, "hidden": 2048, "experts": 128, "top": 8},
        {"name": "router_512", "kind": "router", "rows": 512, "hidden": 2048, "experts": 128, "top": 8},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case of the listed ones' ranges."""
    kind = rng.choice(["decode", "decode", "step", "token", "prefill", "prefill", "prefill", "block", "block",
                       "router"])
    elem = rng.choice(["f16", "f32"])
    if kind == "decode":
        ctx = _log(rng, 33, 32768)
        return {"kind": kind, "layers": _log(rng, 1, min(48, max(1, 131072 // ctx))), "ctx": ctx, "elem": elem}
    if kind == "step":
        return {"kind": kind, "ctx": _log(rng, 1, 16384), "elem": elem}
    if kind == "token":
        return {"kind": kind, "layers": rng.randint(1, 16), "ctx": _log(rng, 1, 4096), "elem": elem,
                "q": rng.choice(["q4", "q5", "q6"]), "v": rng.choice(["q4", "q6"]), "o": rng.choice(["q5", "q6"])}
    if kind == "router":
        return {"kind": kind, "rows": _log(rng, 1, 1024), "hidden": rng.choice([1024, 2048, 4096]),
                "experts": rng.choice([60, 64, 128]), "top": rng.choice([4, 6, 8])}
    mode = rng.choice(["f16", "bf16", "exact"])
    rows = _log(rng, 8, 1024 if kind == "prefill" else 512)
    start = rng.choice([0, _log(rng, 1, 12000 if kind == "prefill" else 4000)])
    if mode == "exact" or elem == "f32":  # no dearer than the largest listed one
        start = min(start, 4000)
    case = {"kind": kind, "mode": mode, "rows": rows, "start": start, "elem": elem}
    if kind == "block":
        case.update(q=rng.choice(["q4", "q5", "q6"]), v=rng.choice(["q4", "q6"]), o=rng.choice(["q5", "q6"]))
    return case


# ---- inputs -----------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)


def _norm_weight(g, n):
    return 1.0 + 0.02 * _randn(g, n)


def _bytes(g, *shape):
    return torch.randint(0, 256, shape, generator=g, device="cuda", dtype=torch.uint8)


def _f16_field(w, off, values):
    w[:, :, off:off + 2] = values.to(torch.float16).unsqueeze(-1).view(torch.uint8)


def _weights(g, fmt, rows, width):
    """Packed rows whose weights spread as a trained projection's do (about 1/sqrt(width) of either sign)."""
    per, size = BLOCK[fmt]
    nb = width // per
    w = _bytes(g, rows, nb, size)
    spread = width ** -0.5 * (0.8 + 0.4 * torch.rand(rows, nb, generator=g, device="cuda"))
    if fmt in ("q4", "q5"):
        levels, std = (15, 4.61) if fmt == "q4" else (31, 9.23)
        sc = torch.randint(16, 64, (rows, nb, 8), generator=g, device="cuda", dtype=torch.uint8)
        lo, hi = sc[:, :, :4], sc[:, :, 4:]
        w[:, :, 4:8] = lo | ((hi >> 4) << 6)   # the six-bit scales and, beside them,
        w[:, :, 8:12] = lo | ((hi >> 4) << 6)  # equal minimum scales: weights centred on 0
        w[:, :, 12:16] = (hi & 15) | ((hi & 15) << 4)
        d = spread / (std * 41.8)
        _f16_field(w, 0, d)
        _f16_field(w, 2, d * (levels / 2))
    elif fmt == "q6":
        sc = torch.randint(24, 128, (rows, nb, 16), generator=g, device="cuda", dtype=torch.int16)
        sign = torch.randint(0, 2, (rows, nb, 16), generator=g, device="cuda", dtype=torch.int16) * 2 - 1
        w[:, :, 192:208] = (sc * sign).to(torch.int8).view(torch.uint8)
        _f16_field(w, 208, spread / (18.5 * 81.0))
    else:
        _f16_field(w, 0, spread / 73.9)
    return w.reshape(-1)


def _block_weights(g, case):
    f = FORMATS
    return B.AttnBlockWeights(
        _norm_weight(g, HIDDEN), f[case["q"]], _weights(g, case["q"], Q_DIM, HIDDEN),
        _weights(g, "q8", KV_DIM, HIDDEN), f[case["v"]], _weights(g, case["v"], KV_DIM, HIDDEN),
        _norm_weight(g, DIM), _norm_weight(g, DIM), f[case["o"]], _weights(g, case["o"], HIDDEN, Q_DIM))


class _Plane:
    """Rows of a cache plane (an address the cache hands out) as a device tensor, which keeps the cache alive."""

    def __init__(self, kv, address, shape, elem):
        self.kv = kv
        self.__cuda_array_interface__ = {"data": (address, False), "shape": shape, "version": 2, "strides": None,
                                         "typestr": "<f2" if elem == "f16" else "<f4"}


def _rows(kv, address, lo, n, elem):
    """Rows lo .. lo + n of a plane."""
    at = address + lo * KV_DIM * (2 if elem == "f16" else 4)
    return torch.as_tensor(_Plane(kv, at, (n, KV_DIM), elem), device="cuda")


def _cache(g, layers, ctx, more, elem):
    """A cache holding ctx rows in every layer with room for `more`, and the views of the rows that come next."""
    kv = rv.KvCache(layers, KV_HEADS, DIM, ctx + more, elem)
    views = []
    for layer in range(layers):
        if ctx:
            kv.append_rows(layer, _randn(g, ctx, KV_DIM), _randn(g, ctx, KV_DIM))
        if more:
            views += [_rows(kv, kv.k_layer(layer)[0], ctx, more, elem), _rows(kv, kv.v_layer(layer)[0], ctx, more, elem)]
    return kv, views


def _captured(once):
    """One token's calls as a graph: an eager pass sizes the workspaces, then the capture."""
    once()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        once()
    return graph


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    s = dict(case)
    if kind == "decode":
        n = case["layers"]
        kv, _ = _cache(g, n, case["ctx"], 0, case["elem"])
        q, out = _randn(g, n, Q_DIM), torch.empty(n, Q_DIM, device="cuda")

        def once():
            for layer in range(n):
                rv.decode_attention(q[layer], kv, layer, SCALE, None, out[layer])

        s.update(kv=kv, q_in=q, out=out, graph=_captured(once))
    elif kind == "step":
        kv, views = _cache(g, 1, case["ctx"], 1, case["elem"])
        s.update(kv=kv, views=views, q_in=_randn(g, Q_DIM), k_in=_randn(g, KV_DIM), v_in=_randn(g, KV_DIM),
                 wq=_norm_weight(g, DIM), wk=_norm_weight(g, DIM), out=torch.empty(Q_DIM, device="cuda"))
    elif kind == "token":
        n = case["layers"]
        kv, views = _cache(g, n, case["ctx"], 1, case["elem"])
        ws = [_block_weights(g, case) for _ in range(n)]
        x = _randn(g, HIDDEN)
        residual = x.clone()
        pos = torch.full((1,), case["ctx"], dtype=torch.int32, device="cuda")
        scratch = torch.empty(max(256, B.scratch_bytes(HIDDEN, Q_DIM, KV_DIM)), dtype=torch.uint8, device="cuda")

        def once():
            residual.copy_(x)
            for layer in range(n):
                B.attn_block_decode_dev(kv, layer, residual, Q_DIM, ws[layer], EPS, THETA, pos, case["ctx"], SCALE,
                                        scratch)

        s.update(kv=kv, views=views, ws=ws, x=x, residual=residual, pos=pos, scratch=scratch, graph=_captured(once))
    elif kind == "prefill":
        n = case["rows"]
        kv, views = _cache(g, 1, case["start"], n, case["elem"])
        s.update(kv=kv, views=views, q_in=_randn(g, n, Q_DIM), k_in=_randn(g, n, KV_DIM), v_in=_randn(g, n, KV_DIM),
                 wq=_norm_weight(g, DIM), wk=_norm_weight(g, DIM), out=torch.empty(n, Q_DIM, device="cuda"))
    elif kind == "block":
        n = case["rows"]
        kv, views = _cache(g, 1, case["start"], n, case["elem"])
        x = _randn(g, n, HIDDEN)
        nbytes = B.prefill_scratch_bytes(n, HIDDEN, Q_DIM, KV_DIM)
        s.update(kv=kv, views=views, w=_block_weights(g, case), x=x, residual=torch.empty_like(x),
                 scratch=torch.empty(max(256, nbytes), dtype=torch.uint8, device="cuda"))
    else:
        n, e, h = case["rows"], case["experts"], case["hidden"]
        s.update(x=_randn(g, n, h), w=_randn(g, e, h) * h ** -0.5,
                 picks=torch.empty(n, case["top"], dtype=torch.int32, device="cuda"),
                 weights=torch.empty(n, case["top"], device="cuda"))
    return s


# ---- one pass -----------------------------------------------------------------

def run(s):
    kind = s["kind"]
    if kind == "decode":
        s["graph"].replay()
        return [s["out"]]
    if kind == "step":
        s["kv"].truncate(s["ctx"])
        rv.decode_step(s["kv"], 0, s["q_in"], s["k_in"], s["v_in"], s["wq"], s["wk"], EPS, THETA, s["ctx"], SCALE,
                       s["out"])
        return [s["out"], *s["views"]]
    if kind == "token":
        s["graph"].replay()
        return [s["residual"], *s["views"]]
    if kind == "prefill":
        s["kv"].truncate(s["start"])
        rv.prefill_chunk(s["kv"], 0, s["q_in"], s["k_in"], s["v_in"], s["wq"], s["wk"], EPS, THETA, s["start"], SCALE,
                         s["out"], s["mode"])
        return [s["out"], *s["views"]]
    if kind == "block":
        s["kv"].truncate(s["start"])
        s["residual"].copy_(s["x"])
        B.attn_block_prefill(s["kv"], 0, s["residual"], Q_DIM, s["w"], EPS, THETA, s["start"], SCALE, s["mode"],
                             s["scratch"])
        return [s["residual"], *s["views"]]
    return list(R.router_topk(s["x"], s["w"], s["top"], True, s["picks"], s["weights"]))


# ---- what a pass cannot do without ------------------------------------------------

def _packed_bytes(fmt, rows, width):
    per, size = BLOCK[fmt]
    return rows * (width // per) * size


def _proj(case, rows):
    """(weight bytes, operations) of the four projections of `rows` rows."""
    b = (_packed_bytes(case["q"], Q_DIM, HIDDEN) + _packed_bytes("q8", KV_DIM, HIDDEN)
         + _packed_bytes(case["v"], KV_DIM, HIDDEN) + _packed_bytes(case["o"], HIDDEN, Q_DIM))
    return b, 2 * rows * (HIDDEN * (Q_DIM + 2 * KV_DIM) + Q_DIM * HIDDEN)


def work(case):
    kind = case["kind"]
    if kind == "router":
        n, e, h = case["rows"], case["experts"], case["hidden"]
        return {"bytes": 4 * (n * h + e * h) + 8 * n * case["top"], "flops": 2 * n * e * h}
    es = 2 if case["elem"] == "f16" else 4
    if kind in ("decode", "step", "token"):
        ctx, layers = case["ctx"], case.get("layers", 1)
        new = 0 if kind == "decode" else 1
        byts = 2 * ctx * KV_DIM * es + new * 2 * KV_DIM * es
        flops = 4 * DIM * (ctx + new) * HEADS
        if kind == "token":
            wb, wf = _proj(case, 1)
            byts, flops = byts + wb + 4 * HIDDEN, flops + wf
            return {"bytes": layers * byts + 8 * HIDDEN, "flops": layers * flops}
        byts += 8 * Q_DIM + new * 8 * KV_DIM
        return {"bytes": layers * byts, "flops": layers * flops}
    n, start = case["rows"], case["start"]
    byts = 2 * start * KV_DIM * es + 2 * n * KV_DIM * es
    flops = 4 * DIM * HEADS * (n * start + n * (n + 1) // 2)
    if kind == "block":
        wb, wf = _proj(case, n)
        return {"bytes": byts + wb + 8 * n * HIDDEN, "flops": flops + wf}
    return {"bytes": byts + 8 * n * Q_DIM + 8 * n * KV_DIM, "flops": flops}


def tolerance(case):
    """About four times the distance to `exact`; for 16-bit cache rows, of the rows to the unrounded ones
    (2.1e-4), the most that flips of their last bit could come to."""
    kind, mode = case["kind"], case.get("mode")
    if kind == "router":
        return {"rel": 6e-6, "differ": 2e-3}
    if kind == "token":  # a step of one quantized attention value moves a layer's outputs
        return {"rel": 2e-3, "max": 0.05}
    if kind == "block":
        return {"rel": {"exact": 1e-3, "f16": 3e-3, "bf16": 1e-2}[mode], "max": 0.1}
    if kind == "prefill" and mode != "exact":
        return {"rel": 1.7e-3 if mode == "f16" else 1.4e-2, "max": 0.1}
    if kind != "decode" and case["elem"] == "f16":
        return {"rel": 2e-5, "max": 2e-3}
    return {"rel": 4e-6 if kind == "prefill" else 1.2e-6, "max": 2e-4}


# ---- the same in 64 bits ----------------------------------------------------------

def _cached(g, ctx, elem):
    """The rows `_cache` appends to one layer, as the cache holds them."""
    if not ctx:
        z = torch.zeros(0, KV_DIM, device="cuda", dtype=torch.float64)
        return z, z
    k, v = _randn(g, ctx, KV_DIM), _randn(g, ctx, KV_DIM)
    return _held(k, elem), _held(v, elem)


def _held(x, elem):
    return (x.to(torch.float16) if elem == "f16" else x.float()).double()


def _rope_norm(x, w, start):
    """Per-head RMSNorm and rotation of rows [n][heads * DIM] at positions start .."""
    n = x.shape[0]
    h = x.double().reshape(n, -1, DIM)
    h = h * torch.rsqrt(h.square().mean(-1, keepdim=True) + EPS) * w.double()
    i = torch.arange(DIM // 2, device="cuda", dtype=torch.float64)
    ang = torch.arange(start, start + n, device="cuda", dtype=torch.float64)[:, None] * THETA ** (-2.0 * i / DIM)
    c, s = ang.cos()[:, None, :], ang.sin()[:, None, :]
    a, b = h[..., :DIM // 2], h[..., DIM // 2:]
    return torch.cat([a * c - b * s, a * s + b * c], -1).reshape(n, -1)


def _attend(q, k, v, start):
    """Causal attention of rows q [n][Q_DIM] at start .. over k, v [start + n][KV_DIM]."""
    n, t = q.shape[0], k.shape[0]
    out = torch.empty(n, HEADS, DIM, device="cuda", dtype=torch.float64)
    qh = q.reshape(n, HEADS, DIM)
    keep = torch.arange(t, device="cuda")[None, :] <= start + torch.arange(n, device="cuda")[:, None]
    for h in range(HEADS):
        at = (h // GROUP) * DIM
        p = (qh[:, h] @ k[:, at:at + DIM].T.contiguous()) * SCALE
        p = torch.softmax(p.masked_fill(~keep, -math.inf), -1)
        out[:, h] = p @ v[:, at:at + DIM].contiguous()
    return out.reshape(n, Q_DIM)


def _unpack(w, fmt, rows, width):
    """Packed rows as float64 [rows][width]."""
    per, size = BLOCK[fmt]
    b = w.reshape(rows, width // per, size)

    def f16(off):
        return b[:, :, off:off + 2].contiguous().view(torch.float16).double()

    if fmt == "q8":
        return (f16(0) * b[:, :, 2:].contiguous().view(torch.int8).double()).reshape(rows, width)
    x = b.to(torch.int32)
    if fmt == "q6":
        parts = []
        for half in range(2):
            qh = x[:, :, 128 + 32 * half:160 + 32 * half]
            for grp in range(4):
                ql = x[:, :, 64 * half + 32 * (grp & 1):64 * half + 32 * (grp & 1) + 32]
                parts.append(((ql >> (4 * (grp >> 1))) & 15) | (((qh >> (2 * grp)) & 3) << 4))
        q = torch.cat(parts, -1).double() - 32.0
        sc = b[:, :, 192:208].contiguous().view(torch.int8).double().repeat_interleave(16, -1)
        return (f16(208) * sc * q).reshape(rows, width)
    five = fmt == "q5"
    qs, parts = x[:, :, 48 if five else 16:], []
    for j in range(8):
        q = (qs[:, :, 32 * (j >> 1):32 * (j >> 1) + 32] >> (4 * (j & 1))) & 15
        parts.append(q | (((x[:, :, 16:48] >> j) & 1) << 4) if five else q)
    q = torch.cat(parts, -1).double()
    s = x[:, :, 4:16]
    sc = torch.cat([s[:, :, :4] & 63, (s[:, :, 8:] & 15) | ((s[:, :, :4] >> 6) << 4)], -1).double()
    m = torch.cat([s[:, :, 4:8] & 63, (s[:, :, 8:] >> 4) | ((s[:, :, 4:8] >> 6) << 4)], -1).double()
    return (f16(0) * sc.repeat_interleave(32, -1) * q - f16(2) * m.repeat_interleave(32, -1)).reshape(rows, width)


def _q8_k(x):
    """Rows through the 256-value activation quantizer and back (its choices are made in 32 bits)."""
    b = x.float().reshape(x.shape[0], -1, 256)
    top = b.gather(-1, b.abs().argmax(-1, keepdim=True))
    inv = torch.where(top != 0, -127.0 / top, torch.zeros_like(top))
    n = (inv * b).round().clamp(-128, 127)
    d = torch.where(top != 0, 1.0 / inv, torch.zeros_like(top))
    return (n.double() * d.double()).reshape(x.shape)


def _q8_0(x):
    b = x.float().reshape(x.shape[0], -1, 32)
    d = b.abs().amax(-1, keepdim=True) / 127.0
    t = b * torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
    n = torch.sign(t) * torch.floor(t.abs() + 0.5)
    return (n.double() * d.to(torch.float16).double()).reshape(x.shape)


def _block(x, w, case, k, v, start, elem):
    """A layer's attention half for rows x [n][HIDDEN]: (residual, new k rows, new v rows)."""
    normed = (x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.attn_norm.double())
    xk, x0 = _q8_k(normed), _q8_0(normed)
    q = xk @ _unpack(w.wq, case["q"], Q_DIM, HIDDEN).T
    kn = x0 @ _unpack(w.wk, "q8", KV_DIM, HIDDEN).T
    vn = xk @ _unpack(w.wv, case["v"], KV_DIM, HIDDEN).T
    kn = _rope_norm(kn, w.k_norm, start)
    k, v = torch.cat([k, _held(kn, elem)]), torch.cat([v, _held(vn, elem)])
    out = _attend(_rope_norm(q, w.q_norm, start), k, v, start)
    return x + _q8_k(out) @ _unpack(w.wo, case["o"], HIDDEN, Q_DIM).T, kn, vn


def exact(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind == "router":
        n, e, h = case["rows"], case["experts"], case["hidden"]
        x, w = _randn(g, n, h), _randn(g, e, h) * h ** -0.5
        p = torch.softmax(x.double() @ w.double().T, -1)
        top = p.topk(case["top"], -1).values
        return [None, top / top.sum(-1, keepdim=True)]
    elem = case["elem"]
    if kind == "decode":
        kvs = [_cached(g, case["ctx"], elem) for _ in range(case["layers"])]
        q = _randn(g, case["layers"], Q_DIM).double()
        return [torch.cat([_attend(q[i:i + 1], k, v, case["ctx"] - 1) for i, (k, v) in enumerate(kvs)])]
    if kind == "token":
        kvs = [_cached(g, case["ctx"], elem) for _ in range(case["layers"])]
        ws = [_block_weights(g, case) for _ in range(case["layers"])]
        x, views = _randn(g, HIDDEN).double()[None], []
        for (k, v), w in zip(kvs, ws):
            x, kn, vn = _block(x, w, case, k, v, case["ctx"], elem)
            views += [kn, vn]
        return [x[0], *views]
    start = case["ctx"] if kind == "step" else case["start"]
    k, v = _cached(g, start, elem)
    if kind == "block":
        x = _randn(g, case["rows"], HIDDEN)  # drawn before the weights below, as in prepare
        return list(_block(x.double(), _block_weights(g, case), case, k, v, start, elem))
    n = case.get("rows", 1)
    q, kn, vn = _randn(g, n, Q_DIM), _randn(g, n, KV_DIM), _randn(g, n, KV_DIM)
    wq, wk = _norm_weight(g, DIM), _norm_weight(g, DIM)
    kn = _rope_norm(kn, wk, start)
    out = _attend(_rope_norm(q, wq, start), torch.cat([k, _held(kn, elem)]), torch.cat([v, _held(vn, elem)]), start)
    return [out[0] if kind == "step" else out, kn, vn.double()]
