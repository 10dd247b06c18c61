"""The work that is timed: one pass each through the public calls of a full-attention layer.

The sizes are the package's own: 24 query heads over 4 KV heads of 256 dims, contexts of 4k to 128k keys, prefill
chunks of 1536 and 2048 rows, speculative blocks of up to 16 rows, the D-LSA read of 4 sinks, a 512-key window and
4096 long-range keys. `draw` spreads the same calls over contexts, row counts, cache modes, head geometries, options
and data types, odd sizes among them.

Where a call appends rows, `run` trims them again afterwards (a host-side length, no device work; what speculative
decoding does with rejected rows), so that every pass sees the same cache.
"""
import math

import numpy as np
import torch

import qw_amd

ROPE_BASE = 1e7
WINDOW, SINK, BLOCK = 512, 4, 512  # the D-LSA read's trailing window and sinks; the keys of a cluster block
GEOMETRIES = ((24, 4, 256), (16, 2, 256), (32, 8, 128), (24, 4, 128))
MODES = ("affine4", "affine8", "int8", "turbo4", "fp16")


def listed():
    g = {"hq": 24, "hkv": 4, "d": 256}
    return [
        # the smallest call of decoding: one token into a short 8-bit context, where latency and launches count
        {"name": "decode_8bit_4k", "kind": "decode", "mode": "affine8", "ctx": 4095, "rows": 1, "rope": False, **g},
        # one token of a long chat out of the QKV projection: RoPE, append and attention over a 4-bit cache
        {"name": "decode_rope_4bit_32k", "kind": "decode", "mode": "affine4", "ctx": 32768, "rows": 1, "rope": True, **g},
        # the same over the served default cache mode, at a document's length that is no multiple of anything
        {"name": "decode_rope_turbo4_100k", "kind": "decode", "mode": "turbo4", "ctx": 100003, "rows": 1, "rope": True, **g},
        # a speculative block of 16 draft tokens, causal within the block
        {"name": "verify_16x64k_4bit", "kind": "decode", "mode": "affine4", "ctx": 65536, "rows": 16, "rope": False, **g},
        # a draft tree: 13 nodes that see the context and their own ancestors, by an explicit mask
        {"name": "verify_tree_13x8k_8bit", "kind": "masked", "mode": "affine8", "ctx": 8190, "rows": 13, "mask": "bool", **g},
        # a prompt's later chunk against its 8-bit cached prefix
        {"name": "prefill_2048x16k_8bit", "kind": "prefill", "mode": "affine8", "ctx": 16384, "rows": 2048, **g},
        # a chunk through the unfused calls: RoPE and relayout, append, and the whole cache back as fp16 rows
        {"name": "append_fetch_2048x6k_4bit", "kind": "fetch", "mode": "affine4", "ctx": 6144, "rows": 2048, **g},
        # a chunk over fp16 K/V that the caller holds itself (views of a larger allocation)
        {"name": "dense_1536x8k", "kind": "dense", "rows": 1536, "ctx": 8192, "softcap": 0.0, "window": 0, **g},
        # the options of sliding-window layers with capped logits, at smaller heads and ragged sizes
        {"name": "dense_window_softcap_1001x5k", "kind": "dense", "rows": 1001, "ctx": 4100, "softcap": 50.0, "window": 4096,
         "hq": 32, "hkv": 8, "d": 128},
        # one sparse decode token at 128k: rank the buckets, expand the picks, append, read the listed rows of the cache
        {"name": "dlsa_decode_128k", "kind": "sparse", "mode": "fp16", "ctx": 131071, "rows": 1, **g},
        # a sparse prefill chunk: each row its sinks, its own window and the chunk's long-range blocks
        {"name": "dlsa_prefill_1536x32k", "kind": "gather", "dtype": "f16", "kv_dtype": "f16", "ctx": 32768, "rows": 1536, "share": 1536, **g},
        # the same read by a bf16 runtime, in a shorter chunk
        {"name": "dlsa_prefill_bf16_512x16k", "kind": "gather", "dtype": "bf16", "kv_dtype": "bf16", "ctx": 16384, "rows": 512, "share": 512, **g},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    hq, hkv, d = rng.choice(GEOMETRIES)
    c = {"hq": hq, "hkv": hkv, "d": d}
    kind = rng.choice(("decode", "decode", "verify", "masked", "prefill", "fetch", "dense", "dense", "sparse", "gather", "gather"))
    if kind in ("decode", "verify"):
        rows = 1 if kind == "decode" else rng.randint(2, 16)
        c.update(kind="decode", mode=rng.choice(MODES), ctx=_log(rng, 256, 131072 if rows == 1 else 65536), rows=rows, rope=rng.random() < 0.5)
    elif kind == "masked":
        c.update(kind=kind, mode=rng.choice(MODES), ctx=_log(rng, 256, 16384), rows=_log(rng, 2, 64), mask=rng.choice(("bool", "f16", "f32")))
    elif kind == "prefill":
        c.update(kind=kind, mode=rng.choice(MODES), ctx=rng.choice((0, _log(rng, 256, 16384))), rows=_log(rng, 64, 2048))
    elif kind == "fetch":
        c.update(kind=kind, mode=rng.choice(MODES), ctx=_log(rng, 64, 8192), rows=_log(rng, 64, 2048))
    elif kind == "dense":
        c.update(kind=kind, rows=_log(rng, 1, 1536), ctx=_log(rng, 64, 8192), softcap=rng.choice((0.0, 0.0, 30.0, 50.0)), window=rng.choice((0, 0, 1024, 4096)))
        if rng.random() < 0.2:
            c["d"] = 64
    elif kind == "sparse":
        c.update(kind=kind, mode=rng.choice(("fp16", "affine8", "affine4")), ctx=_log(rng, 12288, 131072), rows=_log(rng, 1, 16))
    else:
        dt = rng.choice((("f16", "f16"), ("f16", "f16"), ("bf16", "bf16"), ("bf16", "f16"), ("f32", "f32")))
        rows = _log(rng, 16, 1536 if dt == ("f16", "f16") else 384)
        c.update(kind=kind, dtype=dt[0], kv_dtype=dt[1], ctx=_log(rng, 6144, 32768), rows=rows, share=rng.choice((rows, 64, 1)))
    return c


# ------------------------------------------------------------------ inputs

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}


def _generator(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1000003 + case["rows"] * 131 + case["ctx"])
    return g


def _kv(case, g, n):
    """[hkv, n, d] keys and values, N(0, 1) with a scale of its own for each head."""
    out = []
    for _ in range(2):
        s = torch.rand((case["hkv"], 1, 1), device="cuda", generator=g) * 1.5 + 0.5
        out.append((torch.randn((case["hkv"], n, case["d"]), device="cuda", generator=g) * s).half())
    return out


def _long_range(case, g):
    """[rows, 4096] long-range keys: 8 whole blocks from below the first window, drawn once for each `share` rows, ascending."""
    n = (case["ctx"] - WINDOW) // BLOCK - 1
    groups = -(-case["rows"] // case["share"])
    pick = torch.rand((groups, n), device="cuda", generator=g).topk(8, dim=1).indices.sort(dim=1).values + 1
    keys = (pick[:, :, None] * BLOCK + torch.arange(BLOCK, device="cuda")).reshape(groups, -1)
    return keys.repeat_interleave(case["share"], dim=0)[: case["rows"]]


def _inputs(case, seed):
    """The tensors of a case, by name; the same for the timed pass and for its 64-bit value."""
    g = _generator(case, seed)
    kind, hq, hkv, d, rows, ctx = (case[k] for k in ("kind", "hq", "hkv", "d", "rows", "ctx"))
    x = {}
    if kind == "gather":
        dq, dk = DTYPES[case["dtype"]], DTYPES[case["kv_dtype"]]
        x["q"] = torch.randn((1, hq, rows, d), device="cuda", generator=g).to(dq)
        x["k"] = torch.randn((1, hkv, ctx + rows, d), device="cuda", generator=g).to(dk)
        x["v"] = torch.randn((1, hkv, ctx + rows, d), device="cuda", generator=g).to(dk)
        pos = ctx + torch.arange(rows, device="cuda")[:, None]
        parts = [_long_range(case, g), pos - (WINDOW - 1) + torch.arange(WINDOW, device="cuda"), torch.arange(SINK, device="cuda").expand(rows, SINK)]
        x["lists"] = torch.cat(parts, dim=1).to(torch.int32).contiguous()
        x["lengths"] = torch.full((rows,), x["lists"].shape[1], dtype=torch.int32, device="cuda")
        return x
    if kind == "dense":
        n = ctx + rows
        k, v = _kv(case, g, -(-n // 256) * 256)  # the allocation grows in steps; the call sees the rows that are filled
        x["k"], x["v"] = k[None, :, :n], v[None, :, :n]
        x["q"] = torch.randn((1, hq, rows, d), device="cuda", generator=g).half()
        return x
    x["k0"], x["v0"] = _kv(case, g, ctx)
    if case.get("rope") or kind == "fetch":
        x["qkv"] = torch.randn((1, rows, (hq + 2 * hkv) * d), device="cuda", generator=g).half()
        return x
    k, v = _kv(case, g, rows)
    x["k"], x["v"] = k[None], v[None]
    x["q"] = torch.randn((1, hq, rows, d), device="cuda", generator=g).half()
    if kind == "masked":
        # node r's parent is an earlier node: it sees the context, its ancestors and itself
        parent = (torch.rand(rows, device="cuda", generator=g) * torch.arange(rows, device="cuda")).long().tolist()
        tree = np.eye(rows, dtype=bool)
        for r in range(1, rows):
            tree[r] |= tree[parent[r]]
        see = torch.ones((1, 1, rows, ctx + rows), dtype=torch.bool, device="cuda")
        see[0, 0, :, ctx:] = torch.from_numpy(tree).cuda()
        if case["mask"] == "bool":
            x["mask"] = see
        else:
            dt = DTYPES[case["mask"]]
            x["mask"] = torch.zeros(see.shape, dtype=dt, device="cuda").masked_fill_(~see, torch.finfo(dt).min)
    if kind == "sparse":
        # buckets of 8 keys, clustered within each block of 512; scores of one query are near those of the next
        n_b = (ctx + rows) // 8 // 64 * 64
        perm = torch.rand((n_b // 64, BLOCK), device="cuda", generator=g).argsort(dim=1).reshape(-1, 64, 8).sort(dim=2).values
        keys = perm + torch.arange(n_b // 64, device="cuda")[:, None, None] * BLOCK
        x["members"] = torch.full((n_b, 16), -1, dtype=torch.int32, device="cuda")
        x["members"][:, :8] = keys.reshape(n_b, 8).int()
        base = torch.randn((1, n_b), device="cuda", generator=g)
        x["scores"] = (base + 0.3 * torch.randn((rows, n_b), device="cuda", generator=g)).contiguous()
        x["positions"] = ctx + torch.arange(rows, dtype=torch.int32, device="cuda")
    return x


# ------------------------------------------------------------------ the timed pass

def prepare(case, seed):
    x = _inputs(case, seed)
    s = {"case": case, "scale": case["d"] ** -0.5, "x": x}
    if "k0" in x:
        k0, v0 = x.pop("k0"), x.pop("v0")
        cache = qw_amd.KVCache(case["mode"], case["hkv"], case["d"], capacity=case["ctx"] + case["rows"])
        if case["ctx"]:
            cache.update(k0, v0)
        s["cache"] = cache
    if case["kind"] == "sparse":
        s["params"] = qw_amd.DlsaSelectParams(WINDOW, SINK, 4096, 1024, 16, 64)
    return s


def run(s):
    case, x, scale = s["case"], s["x"], s["scale"]
    kind, rows, hq, hkv, d = (case[k] for k in ("kind", "rows", "hq", "hkv", "d"))
    if kind == "gather":
        if case["dtype"] == case["kv_dtype"] == "f16":
            return qw_amd.sparse_attention(x["q"], x["k"], x["v"], x["lists"], x["lengths"], scale)
        return qw_amd.sparse_attention_typed(x["q"], x["k"], x["v"], x["lists"], x["lengths"], scale)
    if kind == "dense":
        return qw_amd.causal_attention(x["q"], x["k"], x["v"], scale, softcap=case["softcap"], window=case["window"])
    cache = s["cache"]
    if kind == "fetch":
        q, k, v = qw_amd.fused_rope_qk_append(x["qkv"], hq, hkv, d, d // 4, ROPE_BASE, positions_base=case["ctx"])
        k, v = cache.update_and_fetch(k, v)
        out = q, k, v
    elif kind == "masked":
        out = cache.update_and_attention(x["q"], x["k"], x["v"], scale, mask=x["mask"])
    elif kind == "sparse":
        lists, lengths, picked, status = qw_amd.dlsa_select(x["scores"], x["members"], x["positions"], x["members"].shape[0], s["params"])
        o = cache.update_and_dlsa_attention(x["q"], x["k"], x["v"], lists, lengths, scale)
        out = o, lists, lengths, picked, status
    elif case.get("rope"):
        out = cache.rope_update_and_attention(x["qkv"], hq, d // 4, ROPE_BASE, scale, causal=rows > 1)
    elif rows > 1:
        out = cache.update_and_causal_attention(x["q"], x["k"], x["v"], scale)
    else:
        out = cache.update_and_attention(x["q"], x["k"], x["v"], scale)
    cache.trim(rows)
    return out


# ------------------------------------------------------------------ what a pass cannot do without

ROW_BYTES = {"affine4": (0.5, 4 / 64), "affine8": (1, 4 / 64), "int8": (1, 2 / 256), "turbo4": (0.5, 3 / 256), "fp16": (2, 0)}


def work(case):
    kind, rows, ctx, hq, hkv, d = (case[k] for k in ("kind", "rows", "ctx", "hq", "hkv", "d"))
    qo = 2 * hq * rows * d * 2
    if kind == "gather":
        es = {"f16": 2, "bf16": 2, "f32": 4}
        w = 8 * BLOCK + WINDOW + SINK
        keys = min(ctx + rows, 8 * BLOCK * -(-rows // case["share"])) + WINDOW + rows + SINK
        return {"bytes": keys * hkv * 2 * d * es[case["kv_dtype"]] + 2 * hq * rows * d * es[case["dtype"]] + rows * w * 4, "flops": 4 * d * hq * rows * w}
    if kind == "dense":
        seen = [min(ctx + r + 1, case["window"] or ctx + rows) for r in range(rows)]
        span = min(ctx + rows, seen[0] + rows - 1)
        return {"bytes": span * hkv * 2 * d * 2 + qo, "flops": 4 * d * hq * sum(seen)}
    per, side = ROW_BYTES[case["mode"]]
    row = hkv * 2 * d * (per + side)
    new = hkv * 2 * rows * d * 2
    if kind == "fetch":
        w = (hq + 2 * hkv) * d * 2 * rows
        return {"bytes": w + hq * rows * d * 2 + ctx * row + rows * row + (ctx + rows) * hkv * 2 * d * 2, "flops": 0}
    if kind == "sparse":
        keys = 4096 + WINDOW + SINK
        n_b = (ctx + rows) // 8 // 64 * 64
        union = min(ctx + rows, 4096 * (1 + 0.1 * (rows - 1)) + WINDOW + rows + SINK)  # neighbouring rows share most of their picks
        return {"bytes": union * row + new + qo + rows * (n_b * 4 + 1024 * 64 + keys * 8), "flops": 4 * d * hq * rows * keys}
    pairs = rows * ctx + (rows * (rows + 1) // 2 if kind != "masked" else rows * rows)
    mask = rows * (ctx + rows) * {"bool": 1, "f16": 2, "f32": 4}[case["mask"]] if kind == "masked" else 0
    return {"bytes": (ctx + rows) * row + new + qo + mask, "flops": 4 * d * hq * pairs}


def tolerance(case):
    """Several times what the pass differs by from its 64-bit value (the figures beside each line)."""
    if case["kind"] == "gather":
        if case["dtype"] == "f32":
            return {"rel": 1e-5}  # sums in 32 bits throughout
        return {"rel": 7e-3} if case["dtype"] == "bf16" else {"rel": 1e-3}  # 1.7e-3 and 2.1e-4: the output's rounding
    if case["kind"] == "sparse":
        return {"rel": 1e-3}  # 2.1e-4; the lists are whole numbers and stay as they are
    if case["kind"] == "fetch":
        return {"rel": 5e-3}  # 1e-4 to 4e-3: a rotated key that rounds to its neighbour moves a code now and then
    return {"rel": 1e-2}  # 0.8e-3 to 6e-3: scores are rounded to fp16 before the softmax, more coarsely the larger they are


# ------------------------------------------------------------------ 64-bit values

def _affine(x, bits):
    """Rows as a group-64 affine cache holds them: f16(f16(code scale) + bias)."""
    n = float(2 ** bits - 1)
    w = x.float().reshape(*x.shape[:-1], -1, 64)
    lo, hi = w.amin(-1, keepdim=True), w.amax(-1, keepdim=True)
    side = lo.abs() > hi.abs()
    scale = ((hi - lo) / n).clamp_min(1e-7)
    scale = torch.where(side, scale, -scale)
    edge = torch.where(side, lo, hi)
    q0 = (edge / scale).round()
    scale, bias = torch.where(q0 != 0, edge / q0, scale), torch.where(q0 != 0, edge, torch.zeros_like(edge))
    code = ((w - bias) / scale).round().clamp(0, n)
    t = (code * scale.half().float()).half()
    return (t.double() + bias.half().double()).half().reshape(x.shape)


def _int8(x):
    s = (x.float().abs().amax(-1, keepdim=True) / 127).half()
    s = torch.where(s > 0, s, torch.ones_like(s))
    code = (x.float() / s.float()).half().float().round().clamp(-127, 127)
    return (code * s.float()).half()


def _signs(n, seed):
    s, out = seed & 0xFFFFFFFF, []
    for _ in range(n):
        s = (1664525 * s + 1013904223) & 0xFFFFFFFF
        out.append(1.0 if s >> 31 else -1.0)
    return torch.tensor(out, dtype=torch.float64, device="cuda")


class _Turbo:
    """The rotated 4-bit codec: signs, Walsh-Hadamard, signs, the nearest of 16 Lloyd-Max centroids of N(0, 1/d)."""

    def __init__(self, d):
        seed = qw_amd.KVCacheMode.DEFAULT_TURBO_SEED
        h = torch.ones((1, 1), dtype=torch.float64, device="cuda")
        while h.shape[0] < d:
            h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
        h = h / math.sqrt(d)
        k = seed + 0x4B5F5345
        self.k = _signs(d, k)[:, None] * h * _signs(d, k + 0x9E3779B9)
        self.v = _signs(d, seed)[:, None] * h * _signs(d, seed + 0x9E3779B9)
        edges = torch.special.ndtri(torch.arange(1, 16, dtype=torch.float64) / 16)
        inf = torch.tensor([math.inf], dtype=torch.float64)
        for _ in range(101):
            lo, hi = torch.cat([-inf, edges]), torch.cat([edges, inf])
            pdf = lambda z: torch.exp(-0.5 * z * z) / math.sqrt(2 * math.pi)  # noqa: E731
            c = (pdf(lo) - pdf(hi)) / (torch.special.ndtr(hi) - torch.special.ndtr(lo))
            edges = (c[1:] + c[:-1]) / 2
        self.c = (c / math.sqrt(d)).float().cuda()

    def index(self, x, basis):
        x = x.double()
        norm = x.norm(dim=-1, keepdim=True)
        y = (x / torch.where(norm > 0, norm, torch.ones_like(norm))) @ basis
        b = ((self.c[1:] + self.c[:-1]) * 0.5).double()
        return torch.bucketize(y, b), norm

    def rotated(self, x, basis):
        """f16(centroid rescale), in the rotated basis."""
        i, norm = self.index(x, basis)
        c = self.c[i]
        r = (norm / c.double().norm(dim=-1, keepdim=True)).half()
        return (c * r.float()).half()

    def fetched_v(self, x):
        i, norm = self.index(x, self.v)
        c = self.c[i].double()
        return ((c / c.norm(dim=-1, keepdim=True)) @ self.v.T) * norm.half().double()


def _rope(x, d, pos0):
    """x [h, rows, d], the first quarter of the dims rotated in half-split pairs."""
    half = d // 8
    inv = torch.exp2(-(torch.arange(half, device="cuda", dtype=torch.float32) / half) * np.float32(np.log2(np.float32(ROPE_BASE))).item())
    th = ((pos0 + torch.arange(x.shape[1], device="cuda")).float()[:, None] * inv[None]).double()
    x, c, s = x.double(), th.cos(), th.sin()
    a, b = x[..., :half], x[..., half : 2 * half]
    return torch.cat([a * c - b * s, a * s + b * c, x[..., 2 * half :]], -1)


def _rows_attention(q, k, v, scale, lo, hi, softcap=0.0, mask=None):
    """fp64 attention of q [hq, L, d] over k, v [hkv, T, d]: row r sees the keys lo[r] <= t < hi[r], plus an additive mask [L, T]."""
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    t = torch.arange(k.shape[1], device="cuda")
    for a in range(0, q.shape[1], 512):
        b = min(q.shape[1], a + 512)
        hidden = (t[None] < lo[a:b, None]) | (t[None] >= hi[a:b, None])
        for h in range(q.shape[0]):
            j = h // (q.shape[0] // k.shape[0])
            s = (q[h, a:b].double() @ k[j].double().T) * scale
            if softcap:
                s = torch.tanh(s / softcap) * softcap
            if mask is not None:
                s = s + mask[a:b]
            out[h, a:b] = torch.softmax(s.masked_fill_(hidden, -math.inf), -1) @ v[j].double()
    return out


def _listed_attention(q, k, v, lists, scale):
    """fp64 attention of each row over the keys of its list, each named once."""
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    for a in range(0, q.shape[1], 512):
        b = min(q.shape[1], a + 512)
        hidden = torch.ones((b - a, k.shape[1] + 1), dtype=torch.bool, device="cuda")
        hidden.scatter_(1, torch.where(lists[a:b] < 0, k.shape[1], lists[a:b]).long(), False)
        hidden = hidden[:, :-1]
        for h in range(q.shape[0]):
            j = h // (q.shape[0] // k.shape[0])
            s = (q[h, a:b].double() @ k[j].double().T) * scale
            out[h, a:b] = torch.softmax(s.masked_fill_(hidden, -math.inf), -1) @ v[j].double()
    return out


def _selected(x, r, p, n):
    """Row r's keys: the members of its best 1024 buckets, its window and the sinks; n fills the rest."""
    seen = min(p // WINDOW * 64, x["members"].shape[0])
    best = torch.sort(x["scores"][r, :seen], descending=True, stable=True).indices[:1024]
    keys = x["members"][best].reshape(-1)
    start = max(0, p + 1 - WINDOW)
    keys = keys[(keys >= SINK) & (keys < start)][:4096]
    keys = torch.cat([keys, torch.arange(start, p + 1, device="cuda"), torch.arange(min(SINK, start), device="cuda")])
    return torch.cat([keys, keys.new_full((4096 + WINDOW + SINK - keys.numel(),), n)])[None]


def exact(case, seed):
    x = _inputs(case, seed)
    kind, rows, ctx, hq, hkv, d = (case[k] for k in ("kind", "rows", "ctx", "hq", "hkv", "d"))
    scale, n = d ** -0.5, ctx + rows
    first = torch.zeros(rows, dtype=torch.long, device="cuda")
    causal = ctx + 1 + torch.arange(rows, device="cuda")
    if kind == "gather":
        return _listed_attention(x["q"][0], x["k"][0], x["v"][0], x["lists"], scale)[None]
    if kind == "dense":
        lo = (causal - case["window"]).clamp_min(0) if case["window"] else first
        return _rows_attention(x["q"][0], x["k"][0], x["v"][0], scale, lo, causal, case["softcap"])[None]
    if "qkv" in x:
        y = x["qkv"][0].reshape(rows, hq + 2 * hkv, d).transpose(0, 1)
        q = _rope(y[:hq], d, ctx)
        k, v = _rope(y[hq : hq + hkv], d, ctx).half(), y[hq + hkv :]
    else:
        q, k, v = x["q"][0], x["k"][0], x["v"][0]
    k, v = torch.cat([x["k0"], k], 1), torch.cat([x["v0"], v], 1)
    mode, out_basis, q_seen = case["mode"], None, q.half()
    if mode == "turbo4":
        turbo = _Turbo(d)
        if kind == "fetch":
            k, v = turbo.rotated(k, turbo.k).double() @ turbo.k.T, turbo.fetched_v(v)
        else:
            q_seen, k, v, out_basis = q_seen.double() @ turbo.k, turbo.rotated(k, turbo.k), turbo.rotated(v, turbo.v), turbo.v.T
    elif mode == "int8":
        k, v = _int8(k), _int8(v)
    elif mode != "fp16":
        k, v = _affine(k, int(mode[-1])), _affine(v, int(mode[-1]))
    if kind == "fetch":
        return q[None], k.double()[None], v.double()[None]
    if kind == "sparse":
        lists = torch.cat([_selected(x, r, ctx + r, n) for r in range(rows)])
        return _listed_attention(q_seen, k, v, lists, scale)[None], None, None, None, None
    mask = None
    if kind == "masked":
        m = x["mask"][0, 0]
        mask = torch.zeros(m.shape, dtype=torch.float64, device="cuda").masked_fill_(~m, -math.inf) if m.dtype == torch.bool else m.half().double()
    hi = causal if rows > 1 and kind != "masked" else torch.full_like(causal, n)
    o = _rows_attention(q_seen, k, v, scale, first, hi, mask=mask)
    o = o if out_basis is None else o @ out_basis
    return (o[None], q[None]) if case.get("rope") else o[None]
