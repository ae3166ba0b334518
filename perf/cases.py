"""What the framework's speed is measured on: the calls a program that serves a quantized model makes.

Kinds of case (the sizes of the listed ones are this repository's own workloads, see each comment in listed()):
  dense     one QMatMul.forward on activations in hand: a lone projection at decode, or a prompt at prefill
  layers    one decode step through a stack of decoder layers' projections, captured once in a HIP graph and
            replayed, as a server does (attention and norms are not this framework's, so their outputs are inputs here)
  mlp       a prompt through one gated MLP: silu(gate) on the store, times up on the store, and the down projection
  moe       one routed SwiGLU layer: silu(gate) * up in one routed call, then the routed down projection
  convert   a weight quantized on the device and read back as numbers, as a program that makes a quantized model does

Weights are blocks in their GGUF layout, quantized from N(0, 0.02) by the plain quantizers below; activations are
N(0, 1) (what a norm hands on) or, into a down projection, products of two normals (what a gated unit hands on).
"""
import math

import torch

from lloom_amd import GgmlDType, QMatMul, QTensor
from lloom_amd.quantized import qmatmul_workspace_bytes, reserve_workspace

DEV = "cuda"
QK = {"q8_0": GgmlDType.Q8_0, "q4k": GgmlDType.Q4K, "q6k": GgmlDType.Q6K}
BLOCK = {"q8_0": (32, 34), "q4k": (256, 144), "q6k": (256, 210)}
ACT = {"f32": torch.float32, "f16": torch.float16}


# ---------------------------------------------------------------- the cases --

def _dense(name, dtype, n, k, m, act="f32"):
    return {"name": name, "kind": "dense", "dtype": dtype, "n": n, "k": k, "m": m, "act": act}


def _layers(name, rows, hidden=2048, kv=512, ffn=8192, count=8):
    return {"name": name, "kind": "layers", "rows": rows, "hidden": hidden, "kv": kv, "ffn": ffn, "count": count}


def _moe(name, tokens, down="q4k", experts=128, topk=8, hidden=2048, ff=768, strict=False):
    return {"name": name, "kind": "moe", "tokens": tokens, "experts": experts, "topk": topk, "hidden": hidden,
            "ff": ff, "down": down, "strict": strict}


def listed():
    return [
        # one token's projection, called eagerly: the smallest call, its launch and host path
        _dense("call_q4k_row", "q4k", 6144, 2048, 1),
        # decode of a 2.6B-class model (hidden 2048, 8 kv heads of 64, FFN 8192; attention and FFN in Q4_K, the down
        # projection in Q6_K): one token, and a full continuous batch; 8 layers are 308 MB of weights, more than
        # the last-level cache holds
        _layers("decode_layers_1", 1),
        _layers("decode_layers_16", 16),
        # the FFN projection of a 70B-class model for a few sequences: a weight far larger than the caches' share
        _dense("large_q4k_rows8", "q4k", 28672, 8192, 8),
        # prompts: a long one, an ordinary ragged one in half precision through the whole MLP, and an 8-bit model's
        _dense("prefill_q4k_2048", "q4k", 8192, 2048, 2048),
        {"name": "mlp_f16_509", "kind": "mlp", "m": 509, "hidden": 2048, "ffn": 8192, "act": "f16"},
        _dense("prefill_q8_0_1000", "q8_0", 8192, 2048, 1000),
        # a mixture of 128 experts, top-8: one token (ids checked before the call returns, the default), a decode
        # batch of 32, a prompt of 512, and a long prompt with the down projection in Q6_K, as mixed files have it
        _moe("moe_token", 1, strict=True),
        _moe("moe_decode_32", 32),
        _moe("moe_prefill_512", 512),
        _moe("moe_prefill_2000_q6k", 2000, down="q6k"),
        # making a quantized model: one FFN weight quantized, and read back
        {"name": "convert_q4k", "kind": "convert", "dtype": "q4k", "n": 8192, "k": 2048},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dense", "dense", "layers", "mlp", "moe", "moe", "convert"])
    if kind == "dense":
        while True:
            c = {"kind": kind, "dtype": rng.choice(["q4k", "q4k", "q6k", "q8_0"]), "n": _log(rng, 300, 28672),
                 "k": 256 * _log(rng, 2, 32), "m": _log(rng, 1, 2300), "act": rng.choice(["f32", "f32", "f16"])}
            if c["n"] * c["k"] * c["m"] <= 8192 * 2048 * 2300:
                return c
    if kind == "layers":
        hidden = 256 * rng.randint(4, 12)
        return {"kind": kind, "rows": rng.randint(1, 16), "hidden": hidden, "kv": 64 * rng.randint(2, 8),
                "ffn": 256 * rng.randint(12, 32), "count": rng.randint(3, 6)}
    if kind == "mlp":
        return {"kind": kind, "m": _log(rng, 17, 1100), "hidden": 256 * rng.randint(4, 12),
                "ffn": 256 * rng.randint(12, 32), "act": rng.choice(["f16", "f32"])}
    if kind == "moe":
        return {"kind": kind, "tokens": _log(rng, 1, 1900), "experts": rng.choice([32, 60, 64, 128]),
                "topk": rng.randint(2, 8), "hidden": 256 * rng.randint(4, 8), "ff": 256 * rng.randint(2, 3),
                "down": rng.choice(["q4k", "q4k", "q6k"]), "strict": rng.random() < 0.25}
    return {"kind": kind, "dtype": rng.choice(["q4k", "q6k", "q8_0"]), "n": _log(rng, 500, 8192),
            "k": 256 * rng.randint(2, 12)}


# ------------------------------------------------- inputs, from the seed alone --

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 1000003 + 17)
    return g


def _f16_bytes(v):
    return v.to(torch.float16).view(torch.uint8).reshape(v.shape[0], 2)


def _blocks_q8_0(w):
    w = w.reshape(-1, 32)
    d = (w.abs().amax(1, keepdim=True) / 127).clamp_min(1e-8)
    q = torch.round(w / d).clamp(-127, 127).to(torch.int8)
    return torch.cat([_f16_bytes(d), q.view(torch.uint8)], 1)


def _blocks_q4k(w):
    w = w.reshape(-1, 8, 32)
    lo = w.amin(2).clamp_max(0.0)
    sc = ((w.amax(2) - lo) / 15).clamp_min(1e-8)
    d = (sc.amax(1, keepdim=True) / 63).to(torch.float16).float().clamp_min(6e-8)
    dm = ((-lo).amax(1, keepdim=True) / 63).to(torch.float16).float().clamp_min(6e-8)
    ls, lm = torch.round(sc / d).clamp(0, 63), torch.round(-lo / dm).clamp(0, 63)
    q = torch.round((w + (dm * lm)[..., None]) / (d * ls).clamp_min(1e-8)[..., None]).clamp(0, 15).to(torch.uint8)
    ls, lm = ls.to(torch.uint8), lm.to(torch.uint8)
    scales = torch.cat([ls[:, :4] | ((ls[:, 4:] >> 4) << 6), lm[:, :4] | ((lm[:, 4:] >> 4) << 6),
                        (ls[:, 4:] & 15) | ((lm[:, 4:] & 15) << 4)], 1)
    qs = (q[:, 0::2] | (q[:, 1::2] << 4)).reshape(-1, 128)
    return torch.cat([_f16_bytes(d), _f16_bytes(dm), scales, qs], 1)


def _blocks_q6k(w):
    w = w.reshape(-1, 16, 16)
    sc = (w.abs().amax(2) / 31).clamp_min(1e-8)
    d = (sc.amax(1, keepdim=True) / 127).to(torch.float16).float().clamp_min(6e-8)
    ls = torch.round(sc / d).clamp(1, 127)
    q = (torch.round(w / (d * ls)[..., None]).clamp(-32, 31) + 32).to(torch.uint8).reshape(-1, 2, 4, 32)
    ql = (q[:, :, :2] & 15) | ((q[:, :, 2:] & 15) << 4)
    h = q >> 4
    qh = h[:, :, 0] | (h[:, :, 1] << 2) | (h[:, :, 2] << 4) | (h[:, :, 3] << 6)
    return torch.cat([ql.reshape(-1, 128), qh.reshape(-1, 64), ls.to(torch.uint8), _f16_bytes(d)], 1)


_MAKE = {"q8_0": _blocks_q8_0, "q4k": _blocks_q4k, "q6k": _blocks_q6k}


def _blocks(g, dtype, rows, k):
    """The packed blocks of a [rows, k] weight on the GPU, made a part at a time."""
    out, step = [], max(1, (1 << 27) // k)
    for r in range(0, rows, step):
        out.append(_MAKE[dtype](torch.randn(min(step, rows - r), k, generator=g, device=DEV) * 0.02))
    return torch.cat(out) if len(out) > 1 else out[0]


def _unblocks(b, dtype):
    """The numbers that blocks stand for, in 64 bits."""
    f = lambda v: v.contiguous().view(torch.float16).double()  # noqa: E731
    if dtype == "q8_0":
        return b[:, 2:].contiguous().view(torch.int8).double() * f(b[:, :2])
    if dtype == "q4k":
        d, dm, s, q = f(b[:, :2]), f(b[:, 2:4]), b[:, 4:16], b[:, 16:].reshape(-1, 4, 32)
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).double() * d
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double() * dm
        q = torch.stack([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()
        return (q * sc[..., None] - mn[..., None]).reshape(-1, 256)
    ql, qh = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 1, 32)
    lo = torch.cat([ql & 15, ql >> 4], 2)
    hi = torch.cat([(qh >> s) & 3 for s in (0, 2, 4, 6)], 2)
    q = (lo | (hi << 4)).reshape(-1, 16, 16).double() - 32
    sc = b[:, 192:208].contiguous().view(torch.int8).double() * f(b[:, 208:])
    return (q * sc[..., None]).reshape(-1, 256)


def _acts(g, shape, act="f32", gated=False):
    x = torch.randn(*shape, generator=g, device=DEV)
    if gated:
        x = x * torch.randn(*shape, generator=g, device=DEV) * 0.5
    return x.to(ACT[act])


def _routing(g, c):
    logits = torch.rand(c["tokens"], c["experts"], generator=g, device=DEV)
    return logits.topk(c["topk"], 1).indices.to(torch.int32)


_PROJ = ("q", "k", "v", "o", "gate", "up", "down")


def _shapes(c):
    h, kv, f = c["hidden"], c["kv"], c["ffn"]
    return {"q": ("q4k", h, h), "k": ("q4k", kv, h), "v": ("q4k", kv, h), "o": ("q4k", h, h),
            "gate": ("q4k", f, h), "up": ("q4k", f, h), "down": ("q6k", h, f)}


def _inputs(c, seed):
    """Everything a case reads: {name: blocks}, with (dtype, shape) beside them, and {name: activations}."""
    g = _gen(seed)
    if c["kind"] == "dense":
        return {"w": (c["dtype"], (c["n"], c["k"]), _blocks(g, c["dtype"], c["n"], c["k"]))}, \
            {"x": _acts(g, (c["m"], c["k"]), c["act"])}
    if c["kind"] == "layers":
        w = {}
        for i in range(c["count"]):
            for p in _PROJ:
                dt, n, k = _shapes(c)[p]
                w["%s%d" % (p, i)] = (dt, (n, k), _blocks(g, dt, n, k))
        return w, {"x": _acts(g, (c["rows"], c["hidden"])), "a": _acts(g, (c["rows"], c["hidden"])),
                   "x2": _acts(g, (c["rows"], c["hidden"])), "f": _acts(g, (c["rows"], c["ffn"]), gated=True)}
    if c["kind"] == "mlp":
        h, f = c["hidden"], c["ffn"]
        w = {"gate": ("q4k", (f, h), _blocks(g, "q4k", f, h)), "up": ("q4k", (f, h), _blocks(g, "q4k", f, h)),
             "down": ("q6k", (h, f), _blocks(g, "q6k", h, f))}
        return w, {"x": _acts(g, (c["m"], h), c["act"]), "f": _acts(g, (c["m"], f), c["act"], gated=True)}
    if c["kind"] == "moe":
        e, h, f = c["experts"], c["hidden"], c["ff"]
        w = {"gate": ("q4k", (e, f, h), _blocks(g, "q4k", e * f, h)), "up": ("q4k", (e, f, h), _blocks(g, "q4k", e * f, h)),
             "down": (c["down"], (e, h, f), _blocks(g, c["down"], e * h, f))}
        return w, {"x": _acts(g, (c["tokens"], 1, h)), "ids": _routing(g, c)}
    return {}, {"src": torch.randn(c["n"], c["k"], generator=g, device=DEV) * 0.02}


# ---------------------------------------------------------------------- calls --

def _layer(m, i, x):
    """One decoder layer's projections: q, k, v, the output projection, the gated unit, the down projection."""
    out = [m["%s%d" % (p, i)].forward(x["x"]) for p in "qkv"]
    out.append(m["o%d" % i].forward(x["a"]))
    return out + _gated(m["gate%d" % i], m["up%d" % i], m["down%d" % i], x["x2"], x["f"])


def _gated(gate, up, down, x, f):
    h = gate.forward_silu(x)
    up.forward_mul_into(x, h)
    return [h, down.forward(f)]


def prepare(case, seed):
    blocks, x = _inputs(case, seed)
    w = {}
    for name in list(blocks):
        dt, shape, b = blocks.pop(name)
        w[name] = QTensor.from_data(b.cpu().numpy().reshape(-1), shape, QK[dt], device=DEV)
        del b
    kind = case["kind"]
    if kind in ("moe", "convert"):
        return {"case": case, "w": w, "x": x}
    m = {name: QMatMul.from_qtensor(t) for name, t in w.items()}
    state = {"case": case, "m": m, "x": x}
    if kind == "layers":
        # the workspace is reserved before the capture, which may not allocate it
        reserve_workspace(max(qmatmul_workspace_bytes(QK[dt], n, k, case["rows"]) for dt, n, k in _shapes(case).values()))
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            state["out"] = [_layer(m, i, x) for i in range(case["count"])]
    return state


def run(state):
    case, x = state["case"], state["x"]
    if case["kind"] == "dense":
        return state["m"]["w"].forward(x["x"])
    if case["kind"] == "layers":
        state["graph"].replay()
        return state["out"]
    if case["kind"] == "mlp":
        m = state["m"]
        return _gated(m["gate"], m["up"], m["down"], x["x"], x["f"])
    if case["kind"] == "moe":
        w = state["w"]
        h = w["gate"].indexed_moe_forward_glu_as(w["up"], x["x"], x["ids"], strict=case["strict"])
        return [h, w["down"].indexed_moe_forward(h, x["ids"], strict=case["strict"])]
    t = QTensor.quantize(x["src"], QK[case["dtype"]])
    return [t.storage[:t.packed_bytes()], t.dequantize()]


# --------------------------------------------------- work, tolerances, 64 bits --

def _weight_bytes(dtype, n, k):
    be, bb = BLOCK[dtype]
    return n * k // be * bb


def work(case):
    c, kind = case, case["kind"]
    if kind == "dense":
        size = 2 if c["act"] == "f16" else 4
        return {"bytes": _weight_bytes(c["dtype"], c["n"], c["k"]) + size * c["m"] * (c["n"] + c["k"]),
                "flops": 2 * c["m"] * c["n"] * c["k"]}
    if kind == "layers":
        r, h, f = c["rows"], c["hidden"], c["ffn"]
        per = [_weight_bytes(dt, n, k) + 4 * r * n for dt, n, k in _shapes(c).values()]
        return {"bytes": c["count"] * (sum(per) - 4 * r * f) + 4 * r * (3 * h + f),  # gate and up give one [r, f]
                "flops": c["count"] * sum(2 * r * n * k for _, n, k in _shapes(c).values())}
    if kind == "mlp":
        m, h, f, size = c["m"], c["hidden"], c["ffn"], 2 if c["act"] == "f16" else 4
        return {"bytes": 2 * _weight_bytes("q4k", f, h) + _weight_bytes("q6k", h, f) + size * m * (2 * h + 2 * f),
                "flops": 6 * m * h * f}
    if kind == "moe":
        t, h, f, e, k = c["tokens"], c["hidden"], c["ff"], c["experts"], c["topk"]
        used = e * (1 - (1 - k / e) ** t)  # experts that some token routes to
        return {"bytes": used * (2 * _weight_bytes("q4k", f, h) + _weight_bytes(c["down"], h, f))
                + 4 * t * (h + k + k * f + k * h), "flops": 6 * t * k * h * f}
    elems = c["n"] * c["k"]
    return {"bytes": 8 * elems + _weight_bytes(c["dtype"], c["n"], c["k"]), "flops": 0}


def tolerance(case):
    if case["kind"] == "convert":
        return "exact"  # bytes, and the numbers they stand for, are the format's own
    if case.get("act") == "f16":
        return {"rel": 1e-3, "max": 2e-3}  # one rounding to 11 bits
    return {"rel": 4e-6, "max": 1e-4}  # 32-bit sums


def _round_away(v):
    v = v.double()
    return torch.trunc(v + torch.copysign(torch.full_like(v, 0.5), v))


def _over(a, b):
    """a / b rounded to 32 bits (a GPU's own 32-bit division need not be)."""
    return (torch.as_tensor(a, dtype=torch.float64, device=DEV) / torch.as_tensor(b, dtype=torch.float64, device=DEV)).float()


def _quantized(x, dtype):
    """The activations as every call reads them: quantized a block at a time (in 32 bits), in 64 bits."""
    x = x.float()
    if dtype == "q8_0":
        b = x.reshape(-1, 32)
        d = _over(b.abs().amax(1, keepdim=True), 127.0)
        inv = torch.where(d != 0, _over(1.0, d), torch.zeros_like(d))
        return (_round_away(b * inv) * d.to(torch.float16).double()).reshape(x.shape)
    b = x.reshape(-1, 256)
    a = b.abs()
    at = torch.where(a == a.amax(1, keepdim=True), torch.arange(256, device=x.device), 256).amin(1, keepdim=True)
    top = b.gather(1, at)
    inv = torch.where(top != 0, _over(-127.0, top), torch.zeros_like(top))
    d = torch.where(inv != 0, _over(1.0, inv), torch.zeros_like(inv))
    return (_round_away(b * inv).clamp(-128, 127) * d.double()).reshape(x.shape)


def _product(w, x):
    dt, (n, k), b = w
    return _quantized(x, dt) @ _unblocks(b, dt).reshape(n, k).T


def _silu(v):
    return v / (1 + torch.exp(-v))


def exact(case, seed):
    if case["kind"] == "convert":
        return None
    w, x = _inputs(case, seed)
    if case["kind"] == "dense":
        return _product(w["w"], x["x"])
    if case["kind"] in ("layers", "mlp"):
        gated = lambda s, a: [_silu(_product(w["gate" + s], a)) * _product(w["up" + s], a),  # noqa: E731
                              _product(w["down" + s], x["f"])]
        if case["kind"] == "mlp":
            return gated("", x["x"])
        return [[_product(w["%s%d" % (p, i)], x["x"]) for p in "qkv"] + [_product(w["o%d" % i], x["a"])]
                + gated(str(i), x["x2"]) for i in range(case["count"])]
    # routed: f32 activations against the dequantized experts, nothing quantized
    e, h, f = case["experts"], case["hidden"], case["ff"]
    ids = x["ids"].long()
    act = x["x"].reshape(-1, h).double()
    hid = torch.empty(*ids.shape, f, dtype=torch.float64, device=DEV)
    out = torch.empty(*ids.shape, h, dtype=torch.float64, device=DEV)
    of = lambda name, i: _unblocks(w[name][2].reshape(e, -1, BLOCK[w[name][0]][1])[i], w[name][0])  # noqa: E731
    for i in range(e):
        t, s = torch.where(ids == i)
        if len(t) == 0:
            continue
        v = _silu(act[t] @ of("gate", i).reshape(f, h).T) * (act[t] @ of("up", i).reshape(f, h).T)
        hid[t, s] = v
        out[t, s] = v @ of("down", i).reshape(h, f).T
    return [hid, out]
