"""The work that a program has this library do, as cases to time and to compare.

A case is one call sequence of a GGUF inference engine's forward pass through
the package's public functions: a projection (or several of one activation) at
decode, speculative-verify and prefill batch sizes, the repacked u4 store's
batched GEMM, and a mixture-of-experts feed-forward step.  The shapes are the
dense model's of the benchmark (hidden 5120, feed-forward 17408, Q5_K attention
projection 7168 x 5120, Q6_K vocabulary head 151936 x 5120), its small
projection (3584 x 1024) and its 256-expert layer; the largest prefill chunk is
512 tokens.  Weights are N(0, 0.02) and activations N(0, 1), encoded here to
GGUF blocks on the device.
"""
import importlib.util
import math
import os
import sys

import torch

Q8_0, Q4_K, Q5_K, Q6_K = 8, 12, 13, 14
TYPES = {"q8_0": Q8_0, "q4_k": Q4_K, "q5_k": Q5_K, "q6_k": Q6_K}
BLOCK = {"q8_0": (32, 34), "q4_k": (256, 144), "q5_k": (256, 176), "q6_k": (256, 210)}
DEV = "cuda"


def _package():
    """The package's directory name is no identifier, so it is loaded by its path."""
    name = "sycl_infer_amd"
    if name not in sys.modules:
        path = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sycl-infer_amd", "__init__.py")
        spec = importlib.util.spec_from_file_location(name, path)
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


# ------------------------------------------------------------------ the cases
def _gemm(type, rows, k, tokens, segs=1, gated=False, residual=False):
    """`segs` matrices of one activation; gated: the activation is silu(gate) * up
    (a down projection); residual: added to the output."""
    return {"kind": "gemm", "type": type, "rows": rows, "k": k, "tokens": tokens, "segs": segs, "gated": gated,
            "residual": residual}


def _u4(rows, k, tokens):
    return {"kind": "u4", "rows": rows, "k": k, "tokens": tokens}


def _moe(tokens, experts, top_k, embd, ff):
    return {"kind": "moe", "tokens": tokens, "experts": experts, "top_k": top_k, "embd": embd, "ff": ff}


def listed():
    return [
        # one token through a small model's projection: latency and the launch itself
        dict(_gemm("q4_k", 3584, 1024, 1), name="small_1"),
        # decode of the dense model's feed-forward, one token: gate and up of one activation
        dict(_gemm("q4_k", 17408, 5120, 1, segs=2), name="gate_up_1"),
        # decode's vocabulary head, one token: the largest matrix
        dict(_gemm("q6_k", 151936, 5120, 1), name="head_1"),
        # speculative verify, 7 tokens: the down projection over silu(gate) * up, onto the residual stream
        dict(_gemm("q4_k", 5120, 17408, 7, gated=True, residual=True), name="down_7"),
        # speculative verify, 7 tokens, on the repacked u4 store
        dict(_u4(17408, 5120, 7), name="u4_up_7"),
        # batched decode, 16 sequences: gate and up of one activation
        dict(_gemm("q4_k", 17408, 5120, 16, segs=2), name="gate_up_16"),
        # batched decode, 16 sequences: router, routed experts and weighted sum of a 256-expert layer
        dict(_moe(16, 256, 8, 2048, 512), name="moe_16"),
        # a short prompt of odd length: gate and up of one activation
        dict(_gemm("q4_k", 17408, 5120, 77, segs=2), name="gate_up_77"),
        # a prompt's ragged last chunk through the fused attention projection
        dict(_gemm("q5_k", 7168, 5120, 200), name="qkv_200"),
        # a prompt's ragged chunk through an 8-bit attention output projection, onto the residual stream
        dict(_gemm("q8_0", 5120, 5120, 333, residual=True), name="attn_out_333"),
        # a full prefill chunk through gate and up, the largest amount of arithmetic
        dict(_gemm("q4_k", 17408, 5120, 512, segs=2), name="gate_up_512"),
        # a full prefill chunk through the Q6_K down projection of a mixed-type model
        dict(_gemm("q6_k", 5120, 17408, 512, gated=True, residual=True), name="down_512"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemm"] * 7 + ["u4", "moe"])
    if kind == "u4":
        return _u4(_log(rng, 1024, 17408), 256 * _log(rng, 4, 68), _log(rng, 1, 32))
    if kind == "moe":
        return _moe(_log(rng, 1, 32), rng.choice([64, 128, 256]), rng.choice([4, 8]), 256 * _log(rng, 4, 16),
                    256 * _log(rng, 2, 6))
    type = rng.choice(["q4_k", "q4_k", "q5_k", "q6_k", "q8_0"])
    rows, k, tokens = _log(rng, 1024, 17408), 256 * _log(rng, 4, 68), _log(rng, 1, 512)
    down = rng.random() < 0.4
    segs = 1 if down else rng.choice([1, 1, 2, 3])
    while segs * rows * k * tokens > 2 * 17408 * 5120 * 512:  # the largest listed one
        rows, k, tokens = rows * 3 // 4, max(1024, k // 512 * 256), tokens * 3 // 4
    return _gemm(type, rows, k, tokens, segs, gated=down and rng.random() < 0.7, residual=down)


def work(case):
    c = case
    if c["kind"] == "gemm":
        qk, qb = BLOCK[c["type"]]
        w = c["segs"] * c["rows"] * (c["k"] // qk) * qb
        x = c["tokens"] * c["k"] * 4 * (2 if c["gated"] else 1)
        q = c["tokens"] * (c["k"] + c["k"] // 32 * 16)                # codes, scales and code sums
        out = c["segs"] * c["tokens"] * c["rows"] * 4 * (2 if c["residual"] else 1)
        return {"bytes": w + x + q + out, "flops": 2 * c["segs"] * c["rows"] * c["k"] * c["tokens"]}
    if c["kind"] == "u4":
        w = c["rows"] * (c["k"] // 2 + c["k"] // 32 * 4)
        x = c["tokens"] * (c["k"] * 4 + 2 * c["k"] + c["k"] // 32 * 6)
        return {"bytes": w + x + c["tokens"] * c["rows"] * 4, "flops": 2 * c["rows"] * c["k"] * c["tokens"]}
    pairs = c["tokens"] * c["top_k"]
    active = c["experts"] * (1 - (1 - c["top_k"] / c["experts"]) ** c["tokens"])  # experts that some token picks, on average
    expert = 3 * c["embd"] * c["ff"] // 256 * 144
    io = c["tokens"] * c["embd"] * 4 * 3 + pairs * c["embd"] * 4 + c["experts"] * c["embd"] * 4 + c["tokens"] * c["experts"] * 4
    return {"bytes": active * expert + io, "flops": 2 * pairs * 3 * c["embd"] * c["ff"] + 2 * c["tokens"] * c["experts"] * c["embd"]}


def tolerance(case):
    # About four times the distance between this path and 64-bit sums of the same
    # quantized operands (fp32 sums).  Codes, ids and code sums are exact.
    if case["kind"] == "moe":
        # the gated product is quantized again between the two expert matrices: a last-bit
        # change of its sums moves a few codes by one
        return {"rel": 1e-4, "max": 2e-2, "differ": 0.0}
    return {"rel": 2e-6, "max": 2e-5, "differ": 0.0}


# ------------------------------------------------------------------ inputs
def _gen(seed, salt):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 1000003 + salt)
    return g


def _normal(shape, seed, salt, scale=1.0):
    return torch.randn(shape, generator=_gen(seed, salt), device=DEV, dtype=torch.float32) * scale


def _f16_bytes(v):
    return v.to(torch.float16).contiguous().view(torch.uint8).reshape(*v.shape, 2)


def _f16(b):
    """[..., 2] bytes of a half -> float64 [...]"""
    return b.contiguous().view(torch.float16).squeeze(-1).double()


def _pack_k4(sc, mn):
    """Eight 6-bit scales and mins -> the 12 scale bytes of a Q4_K / Q5_K block."""
    sc, mn = sc.to(torch.int32), mn.to(torch.int32)
    a = (sc[..., :4] & 63) | ((sc[..., 4:] >> 4) << 6)
    b = (mn[..., :4] & 63) | ((mn[..., 4:] >> 4) << 6)
    c = (sc[..., 4:] & 15) | ((mn[..., 4:] & 15) << 4)
    return torch.cat([a, b, c], -1).to(torch.uint8)


def _encode(type, w):
    """fp32 [rows, k] -> the matrix's GGUF blocks, uint8 [rows, row bytes]: a plain
    minimum / maximum fit per group."""
    n, k = w.shape
    if type == "q8_0":
        g = w.view(n, k // 32, 32)
        d = (g.abs().amax(-1) / 127).to(torch.float16)
        q = torch.round(g / d.float().clamp_min(1e-12)[..., None]).clamp(-127, 127).to(torch.int8).view(torch.uint8)
        return torch.cat([_f16_bytes(d), q], -1).reshape(n, -1)
    nb = k // 256
    if type == "q6_k":
        g = w.view(n, nb, 16, 16)
        at = g.abs().argmax(-1, keepdim=True)
        s = g.gather(-1, at).squeeze(-1) / -32                       # the largest value becomes code -32
        top = s.gather(-1, s.abs().argmax(-1, keepdim=True)).squeeze(-1)
        d = (top / -128).to(torch.float16)
        dd = torch.where(d == 0, torch.ones_like(d), d).float()
        sc = torch.round(s / dd[..., None]).clamp(-128, 127)
        step = dd[..., None] * sc
        step = torch.where(step == 0, torch.ones_like(step), step)
        q = (torch.round(g / step[..., None]).clamp(-32, 31) + 32).to(torch.uint8).view(n, nb, 2, 4, 32)
        ql = torch.cat([(q[..., 0, :] & 15) | ((q[..., 2, :] & 15) << 4), (q[..., 1, :] & 15) | ((q[..., 3, :] & 15) << 4)], -1)
        qh = (q[..., 0, :] >> 4) | ((q[..., 1, :] >> 4) << 2) | ((q[..., 2, :] >> 4) << 4) | ((q[..., 3, :] >> 4) << 6)
        return torch.cat([ql.reshape(n, nb, 128), qh.reshape(n, nb, 64), sc.to(torch.int8).view(torch.uint8), _f16_bytes(d)], -1).reshape(n, -1)
    top = 15 if type == "q4_k" else 31
    g = w.view(n, nb, 8, 32)
    lo = (-g.amin(-1)).clamp_min(0)
    s = (g.amax(-1) + lo) / top
    d, dm = (s.amax(-1) / 63).to(torch.float16), (lo.amax(-1) / 63).to(torch.float16)
    sc = torch.round(s / d.float().clamp_min(1e-12)[..., None]).clamp(0, 63)
    mn = torch.round(lo / dm.float().clamp_min(1e-12)[..., None]).clamp(0, 63)
    step, off = d.float()[..., None] * sc, dm.float()[..., None] * mn
    step = torch.where(step == 0, torch.ones_like(step), step)
    q = torch.round((g + off[..., None]) / step[..., None]).clamp(0, top).to(torch.uint8)
    lo4 = ((q[..., 0::2, :] & 15) | ((q[..., 1::2, :] & 15) << 4)).reshape(n, nb, 128)
    parts = [_f16_bytes(d), _f16_bytes(dm), _pack_k4(sc, mn)]
    if type == "q5_k":
        bit = (q >> 4) << torch.arange(8, device=DEV, dtype=torch.uint8)[:, None]
        parts.append(bit.sum(-2, dtype=torch.int32).to(torch.uint8))
    return torch.cat(parts + [lo4], -1).reshape(n, -1)


def _unpack_k4(b):
    b = b.to(torch.int32)
    s0, s1, s2 = b[..., :4], b[..., 4:8], b[..., 8:12]
    sc = torch.cat([s0 & 63, (s2 & 15) | ((s0 >> 6) << 4)], -1)
    mn = torch.cat([s1 & 63, (s2 >> 4) | ((s1 >> 6) << 4)], -1)
    return sc, mn


def _codes(type, b):
    """A Q4_K / Q5_K matrix's blocks [n, nb, bytes] -> codes [n, nb, 8, 32]"""
    n, nb = b.shape[:2]
    qs = b[..., -128:].view(n, nb, 4, 32)
    q = torch.stack([qs & 15, qs >> 4], -2).reshape(n, nb, 8, 32)
    if type == "q5_k":
        sh = torch.arange(8, device=DEV, dtype=torch.uint8)[:, None]
        q = q | (((b[..., 16:48][..., None, :] >> sh) & 1) << 4)
    return q


def _decode(type, raw):
    """GGUF blocks uint8 [n, row bytes] -> float64 [n, k], exact."""
    n = raw.shape[0]
    qk, qb = BLOCK[type]
    b = raw.view(n, -1, qb)
    nb = b.shape[1]
    if type == "q8_0":
        return (b[..., 2:].contiguous().view(torch.int8).double() * _f16(b[..., :2])[..., None]).reshape(n, -1)
    if type == "q6_k":
        ql, qh = b[..., :128].view(n, nb, 2, 2, 32), b[..., 128:192].view(n, nb, 2, 32)
        q = torch.stack([(ql[..., 0, :] & 15) | ((qh & 3) << 4), (ql[..., 1, :] & 15) | (((qh >> 2) & 3) << 4),
                         (ql[..., 0, :] >> 4) | (((qh >> 4) & 3) << 4), (ql[..., 1, :] >> 4) | ((qh >> 6) << 4)], -2)
        sc = b[..., 192:208].contiguous().view(torch.int8).double() * _f16(b[..., 208:210])[..., None]
        return ((q.reshape(n, nb, 16, 16).double() - 32) * sc[..., None]).reshape(n, -1)
    sc, mn = _unpack_k4(b[..., 4:16])
    step, off = _f16(b[..., :2])[..., None] * sc, _f16(b[..., 2:4])[..., None] * mn
    return (_codes(type, b).double() * step[..., None] - off[..., None]).reshape(n, -1)


CHUNK = 1 << 26  # weights encoded (or decoded to 64 bits) at a time


def _weights(type, rows, k, seed, salt):
    per = max(1, CHUNK // k)
    return torch.cat([_encode(type, _normal((min(per, rows - r), k), seed, salt + 7919 * (r + 1), 0.02)) for r in range(0, rows, per)])


def _gemm_inputs(c, seed):
    x = _normal((c["tokens"], c["k"]), seed, 1)
    up = _normal((c["tokens"], c["k"]), seed, 2) if c["gated"] else None
    res = _normal((c["tokens"], c["rows"]), seed, 3) if c["residual"] else None
    return x, up, res, [_weights(c["type"], c["rows"], c["k"], seed, 10 + i) for i in range(c["segs"])]


def _moe_inputs(c, seed):
    x = _normal((c["tokens"], c["embd"]), seed, 1)
    router = _normal((c["experts"], c["embd"]), seed, 2, 1.0 / math.sqrt(c["embd"]))
    resid = _normal((c["tokens"], c["embd"]), seed, 3)
    banks = [_weights("q4_k", c["experts"] * n, k, seed, 10 + i)
             for i, (n, k) in enumerate([(c["ff"], c["embd"]), (c["ff"], c["embd"]), (c["embd"], c["ff"])])]
    return x, router, resid, banks


def prepare(case, seed):
    """Device buffers, weights and call records that an engine holds for a layer."""
    c, m = case, _package()
    if c["kind"] == "gemm":
        x, up, res, ws = _gemm_inputs(c, seed)
        act = m.alloc_act(c["tokens"], c["k"], DEV)
        outs = [torch.empty((c["tokens"], c["rows"]), device=DEV) for _ in ws]
        segs = [m.make_seg(w, TYPES[c["type"]], c["k"], c["rows"], act, o, c["rows"], residual=res, x=x, act_up=up)
                for w, o in zip(ws, outs)]
        return {"case": c, "m": m, "segs": segs, "act": act, "outs": outs, "held": (x, up, res, ws)}
    if c["kind"] == "u4":
        x = _normal((c["tokens"], c["k"]), seed, 1)
        st = m.w4_pack(_weights("q4_k", c["rows"], c["k"], seed, 10), c["k"], c["rows"])
        act = m.w4_act(x)  # its buffers are filled again by each pass
        return {"case": c, "m": m, "x": x, "st": st, "act": act, "out": torch.empty((c["tokens"], c["rows"]), device=DEV)}
    x, router, resid, banks = _moe_inputs(c, seed)
    M = m.make_moe(*banks, Q4_K, c["embd"], c["ff"], c["experts"])
    return {"case": c, "m": m, "M": M, "x": x, "router": router, "resid": resid, "banks": banks,
            "logits": torch.empty((c["tokens"], c["experts"]), device=DEV), "ws": m.moe_workspace(M, c["tokens"], c["top_k"], DEV),
            "acc": torch.empty((c["tokens"] * c["top_k"], c["embd"]), device=DEV), "out": torch.empty((c["tokens"], c["embd"]), device=DEV)}


def run(state):
    s, m, c = state, state["m"], state["case"]
    if c["kind"] == "gemm":
        if c["segs"] == 1:
            m.quant_gemm(s["segs"][0], c["tokens"])
        else:
            m.quant_gemm_multi(s["segs"], c["tokens"])
        a = s["act"]
        return {"out": s["outs"], "x8": a.x8, "scale": a.xmeta, "sums": a.xsumq}
    if c["kind"] == "u4":
        a = m.w4_act(s["x"], out=s["act"])
        if c["tokens"] == 1:
            m.w4_gemv(s["st"], a, s["out"])
        else:
            m.nat_gemm(s["st"], a, s["out"])
        return {"out": s["out"], "xq": a.xq, "even": a.axe, "odd": a.axo, "asa": a.asa, "xs": a.xs}
    ids, wts = m.moe_route(s["logits"], c["top_k"], x=s["x"], gate_inp=s["router"])
    m.moe_experts(s["M"], s["x"], c["top_k"], ids, s["acc"], s["ws"])
    s["out"].copy_(s["resid"])
    m.moe_reduce(s["acc"], wts, c["top_k"], s["out"])
    return {"out": s["out"], "acc": s["acc"], "ids": ids, "wts": wts, "probs": s["logits"]}


# ------------------------------------------------------------------ 64-bit results
def _trunc_half(v):
    """Non-negative float64 -> the half at or below it, as float64 (subnormals included)."""
    e = torch.floor(torch.log2(v.clamp_min(1e-300))).clamp_min(-14)
    q = torch.exp2(e - 10)
    return torch.floor(v / q) * q


def _silu_mul(x, up):
    # the activation's own arithmetic is fp32, step by step: its bytes are the quantizer's input
    e = torch.exp(-x.double()).float()
    return (x / (1.0 + e)) * up


def _round_away(v):
    return torch.sign(v) * torch.floor(v.abs() + 0.5)


def _quantize(v):
    """fp32 [tokens, k] -> codes float64 [tokens, k/32, 32] and scales float64 [tokens, k/32]: the
    activation format's definition (fp32 steps, the scale truncated to a half)."""
    g = v.view(v.shape[0], -1, 32)
    mx = g.abs().amax(-1)
    top = torch.full_like(mx, 127.0)  # a tensor: division by (or of) a number goes through a rounded reciprocal
    inv = torch.where(mx > 0, top / mx, torch.zeros_like(mx))
    q = _round_away((g * inv[..., None]).double()).clamp(-127, 127)
    return q, _trunc_half((mx / top).double())


def _matmul(x, type, raw):
    """float64 x [t, k] times a matrix's blocks, by chunks of rows: [t, rows]"""
    per = max(1, CHUNK // x.shape[1])
    return torch.cat([x @ _decode(type, raw[r:r + per]).t().contiguous() for r in range(0, raw.shape[0], per)], 1)


def exact(case, seed):
    c = case
    if c["kind"] == "gemm":
        x, up, res, ws = _gemm_inputs(c, seed)
        q, s = _quantize(x if up is None else _silu_mul(x, up))
        xd = (q * s[..., None]).reshape(c["tokens"], c["k"])
        outs = [_matmul(xd, c["type"], w) for w in ws]
        if res is not None:
            outs = [o + res.double() for o in outs]
        scale = torch.stack([s, torch.zeros_like(s)], -1).transpose(0, 1).contiguous()
        return {"out": outs, "x8": None, "scale": scale, "sums": None}
    if c["kind"] == "u4":
        x = _normal((c["tokens"], c["k"]), seed, 1)
        g = x.view(c["tokens"], -1, 32)
        mx = g.abs().amax(-1)
        one = torch.ones_like(mx)
        sc = torch.where(mx > 0, mx / (127.0 * one), one)
        q = _round_away((g * (one / sc)[..., None]).double()).clamp(-127, 127)
        sa = sc.to(torch.float16).double()
        xd = (q * sa[..., None]).reshape(c["tokens"], -1)
        raw = _weights("q4_k", c["rows"], c["k"], seed, 10).view(c["rows"], -1, 144)
        w = []
        for r in range(0, c["rows"], 4096):
            b = raw[r:r + 4096]
            n6, m6 = _unpack_k4(b[..., 4:16])
            step = _trunc_half(_f16(b[..., :2])[..., None] * n6)
            off = _trunc_half(_f16(b[..., 2:4])[..., None] * m6)
            w.append(xd @ (_codes("q4_k", b).double() * step[..., None] - off[..., None]).reshape(b.shape[0], -1).t().contiguous())
        return {"out": torch.cat(w, 1), "xq": None, "even": None, "odd": None, "asa": None, "xs": q.sum(-1)}
    x, router, resid, banks = _moe_inputs(c, seed)
    logits = (x.double() @ router.double().t().contiguous()).float()
    probs = torch.softmax(logits.double(), -1)
    # the order of the fp32 probabilities decides; equal ones go to the lower index
    wts, ids = torch.sort(probs.float(), dim=-1, descending=True, stable=True)
    ids = ids[:, :c["top_k"]]
    top = probs.gather(1, ids)
    wts = top / top.sum(-1, keepdim=True)
    q, s = _quantize(x)
    xd = (q * s[..., None]).reshape(c["tokens"], -1)
    F, E = c["ff"], c["embd"]
    gate, up, down = (b.view(c["experts"], n, -1) for b, n in zip(banks, (F, F, E)))
    acc = torch.empty((c["tokens"], c["top_k"], E), device=DEV, dtype=torch.float64)
    for e in torch.unique(ids).tolist():
        t, j = torch.where(ids == e)
        g, u = xd[t] @ _decode("q4_k", gate[e]).t().contiguous(), xd[t] @ _decode("q4_k", up[e]).t().contiguous()
        hq, hs = _quantize(_silu_mul(g.float(), u.float()))
        acc[t, j] = (hq * hs[..., None]).reshape(len(t), -1) @ _decode("q4_k", down[e]).t().contiguous()
    out = resid.double() + (acc * wts[..., None]).sum(1)
    return {"out": out, "acc": acc.reshape(-1, E), "ids": None, "wts": wts, "probs": probs}
