"""The calls that a program built on this package makes, with their sizes: what a speed measurement
of the quantized-matmul path runs.

Each case is one public entry point (gemv, GemvBatch, gate_up_act, logits, MoeLayer) on data that a
model has at that point: weights drawn N(0, 0.02) and packed by the package's own quantizers,
activations N(0, 1) in F32.  Weights are held in the layout that the program holds them in: repacked
once at load (X8, SPLIT, TILE64), or as they lie in the GGUF file.  Outputs and workspaces that a
serving loop keeps are made once, outside the pass.
"""
import math

import torch

import syntropy_amd.gemv as S
import syntropy_amd.moe as M

TYPES = {"F16": S.WeightType.F16, "BF16": S.WeightType.BF16, "Q4_0": S.WeightType.Q4_0,
         "Q8_0": S.WeightType.Q8_0, "Q4_K": S.WeightType.Q4K}
BLOCK = {"F16": (1, 2), "BF16": (1, 2), "Q4_0": (32, 18), "Q8_0": (32, 34), "Q4_K": (256, 144)}
SEGMENTS = 1 << 24  # values packed by the quantizer; a larger matrix repeats their blocks in random order
EPS = 1e-5


def listed():
    return [
        # one small matrix against one token: a single launch, its latency and its fixed cost
        {"name": "row_q4_0", "op": "gemv", "type": "Q4_0", "layout": "packed", "n": 4096, "k": 4096, "rows": 1},
        # all matrices of one decoder layer of an 8B model, one token (QKV, O, gate, up, down), grouped
        {"name": "decode_layer_q4_k", "op": "layer", "type": "Q4_K", "layout": "packed", "hidden": 4096, "kv": 1024,
         "inter": 14336},
        # the gate/up half of that layer's FFN for a few sequences decoded together
        {"name": "ffn_q4_k_6_rows", "op": "gate_up", "type": "Q4_K", "layout": "packed", "n": 14336, "k": 4096,
         "rows": 6},
        # the 8-bit FFN up-projection for a batch of sequences decoded together
        {"name": "batch_q8_0_32_rows", "op": "gemv", "type": "Q8_0", "layout": "packed", "n": 14336, "k": 4096,
         "rows": 32},
        # the half-precision output head over a batch of sequences' last tokens
        {"name": "head_f16_9_rows", "op": "logits", "type": "F16", "layout": "gguf", "n": 32064, "k": 4096, "rows": 9},
        # a long prompt through the 4-bit FFN up-projection
        {"name": "prefill_q4_k_2048", "op": "gemv", "type": "Q4_K", "layout": "packed", "n": 14336, "k": 4096,
         "rows": 2048},
        # a short prompt of odd length through the gate/up pair of a narrower model, weights as in the file
        {"name": "prefill_q4_k_333_gguf", "op": "gate_up", "type": "Q4_K", "layout": "gguf", "n": 5632, "k": 2048,
         "rows": 333},
        # a medium prompt through the 8-bit FFN down-projection
        {"name": "prefill_q8_0_512", "op": "gemv", "type": "Q8_0", "layout": "packed", "n": 4096, "k": 14336,
         "rows": 512},
        # a short prompt over 4-bit weights as they lie in the file, none repacked
        {"name": "prefill_q4_0_200_gguf", "op": "gemv", "type": "Q4_0", "layout": "gguf", "n": 6144, "k": 4096,
         "rows": 200},
        # a large MoE layer, 64 sequences decoded together (route, pack, experts, combine)
        {"name": "moe_q4_k_decode_64", "op": "moe", "type": "Q4_K", "layout": "packed", "experts": 128, "top_k": 8,
         "hidden": 4096, "inter": 1536, "rows": 64, "skew": 0},
        # the same layer over a long prompt with three experts far above the average load
        {"name": "moe_q4_k_prefill_2048", "op": "moe", "type": "Q4_K", "layout": "packed", "experts": 128, "top_k": 8,
         "hidden": 4096, "inter": 1536, "rows": 2048, "skew": 3},
        # a smaller MoE layer with 8-bit experts over a short prompt
        {"name": "moe_q8_0_prefill_300", "op": "moe", "type": "Q8_0", "layout": "gguf", "experts": 64, "top_k": 6,
         "hidden": 2048, "inter": 1408, "rows": 300, "skew": 0},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _width(rng, lo, hi, unit):
    return unit * _log(rng, max(1, lo // unit), hi // unit)


def draw(rng):
    """A case of the same kinds: any listed entry point, type and layout, sizes from small models to
    large ones, row counts from one token to a long prompt."""
    op = rng.choice(["gemv", "gemv", "gemv", "layer", "gate_up", "logits", "moe"])
    if op == "layer":
        hidden = _width(rng, 1024, 5120, 256)
        return {"op": op, "type": "Q4_K", "layout": "packed", "hidden": hidden, "kv": 256 * rng.randint(1, 5),
                "inter": _width(rng, 2 * hidden, min(16384, 4 * hidden), 256)}
    if op == "moe":
        ty = rng.choice(["Q4_K", "Q4_K", "Q8_0"])
        unit = 256 if ty == "Q4_K" else 32
        tile = ty == "Q4_K" and rng.random() < 0.7
        experts = rng.choice([8, 16, 32, 64, 128])
        return {"op": op, "type": ty, "layout": "packed" if tile else "gguf", "experts": experts,
                "top_k": rng.randint(1, min(8, experts)), "hidden": 256 * rng.randint(4, 16),
                "inter": _width(rng, 512, 1536, unit), "rows": _log(rng, 1, 1024 if ty == "Q4_K" else 512),
                "skew": rng.choice([0, 0, 2])}
    ty = rng.choice(["Q4_K", "Q4_K", "Q8_0", "Q8_0", "Q4_0", "F16", "BF16"])
    layout = "gguf" if ty in ("F16", "BF16") or rng.random() < 0.3 else "packed"
    rows = _log(rng, 1, {"F16": 32, "BF16": 32}.get(ty, 256 if layout == "gguf" and ty != "Q4_K" else 1024))
    if ty == "Q4_K":  # X8 rows are whole runs of eight super-blocks from 32 rows on
        k = _width(rng, 1024, 14336, 2048 if layout == "packed" and rows >= 32 else 256)
    else:
        k = _width(rng, 1024, 14336 if op == "gemv" else 8192, 32)
    if op == "logits":
        n, k, rows = _log(rng, 8000, 40000), min(k, 6144), min(rows, 64)
    else:
        n = _log(rng, 512, 14336)
    if op == "gate_up":
        n = max(256, n // 2)
    return {"op": op, "type": ty, "layout": layout, "n": n, "k": k, "rows": rows}


# ---- inputs ---------------------------------------------------------------------------------------

def _gen(seed, part):
    g = torch.Generator(device="cuda")
    g.manual_seed(1_000_003 * (int(seed) % (1 << 40)) + part)
    return g


def _normal(seed, part, *shape):
    return torch.randn(*shape, generator=_gen(seed, part), device="cuda", dtype=torch.float32)


def _bytes(ty, n, k, seed, part):
    """An n x k matrix of type ty in GGUF order, as bytes."""
    elems, size = BLOCK[ty]
    blocks = n * k // elems
    some = min(blocks, SEGMENTS // elems)
    w = _normal(seed, part, some * elems) * 0.02
    if ty in ("F16", "BF16"):
        p = w.to(torch.float16 if ty == "F16" else torch.bfloat16).view(torch.uint8).view(some, size)
        p, blocks, some = p.view(-1, 64), blocks * size // 64, some * size // 64
        rest = n * k * size - blocks * 64
    else:
        p, rest = S.quantize(TYPES[ty], w).view(some, size), 0
    if blocks > some:
        at = torch.randint(some, (blocks,), generator=_gen(seed, part + 500), device="cuda")
        p = p[at]
    p = p[:blocks].reshape(-1)
    return torch.cat([p, p[:rest]]) if rest else p


def _weights(c, n, k, seed, part):
    w = S.Weights(TYPES[c["type"]], _bytes(c["type"], n, k, seed, part), n, k)
    return S.repack(w) if c["layout"] == "packed" else w


def _layer_shapes(c):
    h, i = c["hidden"], c["inter"]
    return [(h + 2 * c["kv"], h), (h, h), (i, h), (i, h), (h, i)]


def _router(c, seed):
    r = _normal(seed, 1, c["experts"], c["hidden"]) * 0.02
    for e in range(c["skew"]):  # popular experts
        r[(3 + 47 * e) % c["experts"]] *= 3.0
    return r


def _experts(c, seed):
    s = M.MoeShape(c["experts"], c["top_k"], c["hidden"], c["inter"])
    mats = [_bytes(c["type"], c["experts"] * n, k, seed, 10 + i)
            for i, (n, k) in enumerate([(s.inter, s.hidden), (s.inter, s.hidden), (s.hidden, s.inter)])]
    return s, M.Experts(TYPES[c["type"]], *mats)


def _tiled(c):
    return c["type"] == "Q4_K" and c["layout"] == "packed" and (c["inter"] % 64 == 0 and c["hidden"] % 64 == 0)


def prepare(case, seed):
    c = case
    if c["op"] == "moe":
        s, experts = _experts(c, seed)
        if _tiled(c):
            experts = M.tile64(experts, s)
        return {"layer": M.MoeLayer(s, _router(c, seed), experts, c["rows"]),
                "x": _normal(seed, 2, c["rows"], c["hidden"]), "c": c}
    if c["op"] == "layer":
        shapes = _layer_shapes(c)
        ws = [_weights(c, n, k, seed, 10 + i) for i, (n, k) in enumerate(shapes)]
        xs = [_normal(seed, 2 + i, k) for i, (_, k) in enumerate(shapes)]
        ys = [torch.empty(n, device="cuda", dtype=torch.float32) for n, _ in shapes]
        return {"batch": S.GemvBatch(ws, xs, ys), "ys": ys, "c": c}
    n = 2 * c["n"] if c["op"] == "gate_up" else c["n"]
    st = {"w": _weights(c, n, c["k"], seed, 10), "x": _normal(seed, 2, c["rows"], c["k"]),
          "y": torch.empty(c["rows"], c["n"], device="cuda", dtype=torch.float32), "c": c}
    if c["op"] == "logits":
        st["g"] = 1.0 + 0.1 * _normal(seed, 3, c["k"])
    return st


def run(state):
    c = state["c"]
    if c["op"] == "moe":
        return state["layer"](state["x"])
    if c["op"] == "layer":
        state["batch"]()
        return state["ys"]
    if c["op"] == "gate_up":
        return S.gate_up_act(state["w"], state["x"], c["rows"], y=state["y"])
    if c["op"] == "logits":
        return S.logits(state["w"], state["g"], EPS, state["x"], c["rows"], y=state["y"])
    return S.gemv(state["w"], state["x"], c["rows"], y=state["y"])


def work(case):
    c = case
    elems, size = BLOCK[c["type"]]
    if c["op"] == "layer":
        shapes = _layer_shapes(c)
        return {"bytes": sum(n * k // elems * size + 4 * (n + k) for n, k in shapes),
                "flops": sum(2 * n * k for n, k in shapes)}
    if c["op"] == "moe":
        e, t, r = c["experts"], c["top_k"], c["rows"]
        used = e * (1 - (1 - t / e) ** r)  # experts that some token is routed to, on average
        mat = c["hidden"] * c["inter"]
        # the router, the used experts' three matrices, x; every slot's output, y, ids and weights
        return {"bytes": 4 * e * c["hidden"] + used * 3 * mat // elems * size + 4 * r * c["hidden"] * (2 + t) + 8 * r * t,
                "flops": 6 * r * t * mat + 2 * r * e * c["hidden"]}
    n = 2 * c["n"] if c["op"] == "gate_up" else c["n"]
    return {"bytes": n * c["k"] // elems * size + 4 * c["rows"] * (c["k"] + c["n"]), "flops": 2 * n * c["k"] * c["rows"]}


def tolerance(case):
    return TOL[case["op"]]


# Sums of F32 terms in another order, about four times what a pass differs by from its 64-bit value;
# the MoE layer's rows are quantized to 8 bits between its products, where a last-bit difference can
# move a code, and a near-tie of the router's logits can exchange two experts.
TOL = {"gemv": {"rel": 2e-6, "max": 1.2e-5}, "layer": {"rel": 2e-6, "max": 1.2e-5},
       "gate_up": {"rel": 2e-6, "max": 1.2e-5}, "logits": {"rel": 2e-6, "max": 1.2e-5},
       "moe": {"rel": 5e-4, "max": 5e-2, "differ": 1e-3}}


# ---- the same in 64 bits ----------------------------------------------------------------------------

def _f16(b):
    return b.contiguous().view(torch.float16).to(torch.float64)


def _dense(ty, raw, n, k):
    """The matrix's values in 64 bits from its GGUF bytes."""
    elems, size = BLOCK[ty]
    if ty in ("F16", "BF16"):
        return raw.view(torch.float16 if ty == "F16" else torch.bfloat16).view(n, k).to(torch.float64)
    b = raw.view(-1, size)
    if ty == "Q8_0":
        return (_f16(b[:, :2]) * b[:, 2:].contiguous().view(torch.int8).to(torch.float64)).view(n, k)
    if ty == "Q4_0":
        q = torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).to(torch.float64) - 8.0
        return (_f16(b[:, :2]) * q).view(n, k)
    d, dmin, s = _f16(b[:, 0:2]), _f16(b[:, 2:4]), b[:, 4:16]
    sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).to(torch.float64)
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).to(torch.float64)
    q = b[:, 16:].view(-1, 4, 32)
    q = torch.stack([q & 15, q >> 4], 2).view(-1, 8, 32).to(torch.float64)
    return ((d * sc).unsqueeze(2) * q - (dmin * mn).unsqueeze(2)).view(n, k)


def _act(ty, x):
    """The rows as the product takes them, in 64 bits: F32 as they are, else their 8-bit blocks (whose
    scale and codes are defined by F32 steps)."""
    if ty in ("F16", "BF16"):
        return x.to(torch.float64)
    x = x.to(torch.float32)
    rows, k = x.shape
    if ty == "Q4_K":
        v = x.view(-1, 256)
        mx = v.gather(1, v.abs().argmax(1, keepdim=True))
        scale = torch.full_like(mx, -127.0) / mx
        q = torch.clamp(torch.round(scale * v), max=127.0)
        d = torch.ones_like(scale) / scale
    else:
        v = x.view(-1, 32)
        d = v.abs().amax(1, keepdim=True) / torch.full_like(v[:, :1], 127.0)
        q = torch.round(v * (torch.ones_like(d) / d))
        d = d.to(torch.float16)
    return (q.to(torch.float64) * d.to(torch.float64)).view(rows, k)


def _silu(x):
    return x / (1.0 + torch.exp(-x))


def _moe_exact(c, seed):
    s, ex = _experts(c, seed)
    x = _normal(seed, 2, c["rows"], c["hidden"])
    p = torch.softmax(x.to(torch.float64) @ _router(c, seed).to(torch.float64).T, 1)
    w, ids = torch.topk(p, c["top_k"], 1)
    w = w / w.sum(1, keepdim=True)
    xq = _act(c["type"], x)
    out = torch.zeros(c["rows"], c["top_k"], c["hidden"], dtype=torch.float64, device="cuda")
    for e in range(c["experts"]):
        row, slot = (ids == e).nonzero(as_tuple=True)
        if not len(row):
            continue
        g, u, dn = (_dense(c["type"], t.view(c["experts"], -1)[e], n, k) for t, n, k in
                    ((ex.gate, s.inter, s.hidden), (ex.up, s.inter, s.hidden), (ex.down, s.hidden, s.inter)))
        h = _silu(xq[row] @ g.T) * (xq[row] @ u.T)
        out[row, slot] = _act(c["type"], h) @ dn.T
    return (out * w.unsqueeze(2)).sum(1), None, w, out


def exact(case, seed):
    c = case
    if c["op"] == "moe":
        return _moe_exact(c, seed)
    if c["op"] == "layer":
        return [(_act(c["type"], _normal(seed, 2 + i, 1, k)) @ _dense(c["type"], _bytes(c["type"], n, k, seed, 10 + i), n, k).T)[0]
                for i, (n, k) in enumerate(_layer_shapes(c))]
    n = 2 * c["n"] if c["op"] == "gate_up" else c["n"]
    x = _normal(seed, 2, c["rows"], c["k"])
    if c["op"] == "logits":
        g = 1.0 + 0.1 * _normal(seed, 3, c["k"])
        x = x.to(torch.float64)
        x = x / torch.sqrt((x * x).mean(1, keepdim=True) + EPS) * g.to(torch.float64)
    y = _act(c["type"], x) @ _dense(c["type"], _bytes(c["type"], n, c["k"], seed, 10), n, c["k"]).T
    return _silu(y[:, :c["n"]]) * y[:, c["n"]:] if c["op"] == "gate_up" else y
