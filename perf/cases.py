"""The work a user of this library has it do, as measurable cases.

Every case goes through the public Python entry points (mlxq.py, stack.py) on
device tensors: quantized projections at decode, batched-decode and prefill
row counts, quantizing and dequantizing weights, decoding and converting GGUF
tensors, and a whole decode step.  `listed()` names the cases, `draw()` takes
one more from the ranges they stand for, `prepare()` makes what a program
holds before the call from a seed alone, `run()` is one pass, `exact()` the
same pass in float64 with plain torch.
"""
from __future__ import annotations

import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mlx-llm_amd"))
import mlxq  # noqa: E402
import stack  # noqa: E402

DEV = "cuda"
BF16, F32, F64 = torch.bfloat16, torch.float32, torch.float64

# (hidden, intermediate, key/value width) of decoder layers: the benchmark's
# 8-billion-parameter shape first, then common sizes around it
LAYERS = [(4096, 14336, 1024), (2048, 5632, 256), (3072, 8192, 1024), (4096, 11008, 4096), (5120, 13824, 1024)]
HEAD = 128  # head size (q/k un-permute, head repeat)
PROJ = ("q", "k", "v", "o", "gate", "up", "down")
# (attention and gate/up type, value and down type) of GGUF files: the k-quant
# mixes, the plain formats and unquantized files
MIXES = [("Q4_K", "Q6_K"), ("Q5_K", "Q6_K"), ("Q3_K", "Q5_K"), ("Q2_K", "Q3_K"), ("Q4_0", "Q4_0"), ("Q5_0", "Q5_0"),
         ("Q8_0", "Q8_0"), ("IQ4_NL", "IQ4_NL"), ("IQ4_XS", "Q5_K"), ("F16", "F16"), ("BF16", "BF16")]


def listed():
    h, i, kv = LAYERS[0]
    dims = {"hidden": h, "inter": i, "kv": kv}
    return [
        # one projection called eagerly for one token: the smallest call, latency
        {"name": "linear_q4_m1", "kind": "linear", "m": 1, "n": kv, "k": h, "bits": 4, "gs": 64, "bias": False},
        # the seven projections of a decoder layer for one token, captured in a
        # graph as decode loops hold them: 4-bit single-user decoding
        {"name": "layer_q4_m1", "kind": "layer", "m": 1, "bits": 4, "gs": 64, **dims},
        # the same for a few sequences on 8-bit weights
        {"name": "layer_q8_m4", "kind": "layer", "m": 4, "bits": 8, "gs": 64, **dims},
        # the same for a server's full decode batch
        {"name": "layer_q4_m32", "kind": "layer", "m": 32, "bits": 4, "gs": 64, **dims},
        # a short prompt of no round length through a layer's projections
        {"name": "prefill_q4_m333", "kind": "prefill", "m": 333, "bits": 4, "gs": 64, **dims},
        # a long prompt: the matrix-core bound end
        {"name": "prefill_q4_m2048", "kind": "prefill", "m": 2048, "bits": 4, "gs": 64, **dims},
        # quantize-on-load of a dense checkpoint's MLP matrix
        {"name": "quantize_bf16_q4", "kind": "quantize", "rows": i, "cols": h, "dtype": "bf16", "bits": 4, "gs": 64},
        # the dense weight of an 8-bit matrix back
        {"name": "dequantize_q8_bf16", "kind": "dequantize", "rows": h, "cols": i, "dtype": "bf16", "bits": 8,
         "gs": 64},
        # a layer of a 4-bit k-quant GGUF file decoded to f32
        {"name": "gguf_q4k_f32", "kind": "gguf_dequant", "main": "Q4_K", "down": "Q6_K", "dtype": "f32", **dims},
        # a layer of a 5-bit k-quant GGUF file decoded to bf16 (a dense conversion)
        {"name": "gguf_q5k_bf16", "kind": "gguf_dequant", "main": "Q5_K", "down": "Q6_K", "dtype": "bf16", **dims},
        # a layer of a 4-bit k-quant GGUF file converted to packed 4-bit weights
        {"name": "convert_q4k_q4", "kind": "gguf_convert", "main": "Q4_K", "down": "Q6_K", "bits": 4, "gs": 64,
         **dims},
        # a whole decode step for one token: embedding row in, logits out
        {"name": "step_q4_b1", "kind": "step", "m": 1, "layers": 4, "vocab": 128256, "bits": 4, "gs": 64, **dims},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(lo * (hi / lo) ** rng.random())))


def draw(rng):
    kind = rng.choice(["linear", "layer", "layer", "prefill", "prefill", "quantize", "dequantize", "gguf_dequant",
                       "gguf_dequant", "gguf_convert", "gguf_convert", "step"])
    bits, gs = rng.choice([4, 4, 8]), rng.choice([64, 64, 64, 32, 128])
    h, i, kv = rng.choice(LAYERS)
    dims = {"hidden": h, "inter": i, "kv": kv}
    if kind == "linear":
        return {"kind": kind, "m": _log_int(rng, 1, 64), "n": _log_int(rng, 65, 16384), "k": 128 * _log_int(rng, 4, 112),
                "bits": bits, "gs": gs, "bias": rng.random() < 0.5}
    if kind == "layer":
        return {"kind": kind, "m": _log_int(rng, 1, 32), "bits": bits, "gs": gs, **dims}
    if kind == "prefill":
        return {"kind": kind, "m": _log_int(rng, 33, 1536), "bits": bits, "gs": gs, **dims}
    if kind in ("quantize", "dequantize"):
        n, k = rng.choice([(i, h), (h, i), (h, h), (kv, h)])
        return {"kind": kind, "rows": max(1, n - rng.randrange(0, 64)), "cols": k, "dtype": rng.choice(["bf16", "f32"]),
                "bits": bits, "gs": gs}
    main, down = rng.choice(MIXES)
    if kind == "gguf_dequant":
        return {"kind": kind, "main": main, "down": down, "dtype": rng.choice(["f32", "bf16"]), **dims}
    if kind == "gguf_convert":
        return {"kind": kind, "main": main, "down": down, "bits": bits, "gs": gs, **dims}
    return {"kind": "step", "m": _log_int(rng, 1, 32), "layers": rng.randint(1, 4),
            "vocab": rng.choice([32000, 32003, 128256]), "bits": bits, "gs": 64, **dims}


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=F32)


def _group_params(w, gs, bits):
    """(scale f32, bias f32) [N, K/gs] of the group-wise affine rule: the
    edge of larger magnitude is the bias, the scale puts 0 on the grid."""
    t = w.float().view(w.shape[0], -1, gs)
    hi, lo = t.amax(2), t.amin(2)
    bins = torch.full_like(hi, 2**bits - 1)  # a tensor: dividing by a number would multiply by its reciprocal
    neg = lo.abs() > hi.abs()
    scale = torch.clamp((hi - lo) / bins, min=1e-7)
    scale = torch.where(neg, scale, -scale)
    edge = torch.where(neg, lo, hi)
    q0 = torch.round(edge / scale)
    return edge, q0, scale


def _pack(q, bits):
    """Integer codes [N, K] -> int32 words [N, K * bits / 32], low bits first."""
    per = 32 // bits
    q = q.to(torch.int32).view(q.shape[0], -1, per)
    out = q[..., 0].clone()
    for j in range(1, per):
        out |= q[..., j] << (bits * j)
    return out


def _qlinear(g, n, k, gs, bits):
    """Packed weights of a seeded N(0, 0.02) matrix: (wq, scales, biases)."""
    w = _randn(g, n, k).mul_(0.02).to(BF16)
    edge, q0, scale = _group_params(w, gs, bits)
    scale = torch.where(q0 != 0, edge / q0, scale)
    bias = torch.where(q0 != 0, edge, torch.zeros_like(edge))
    q = ((w.float().view(n, -1, gs) - bias[..., None]) / scale[..., None]).round_().clamp_(0, 2**bits - 1)
    return _pack(q.view(n, k), bits), scale.to(BF16), bias.to(BF16)


def _dense64(wq, s, b, gs, bits):
    """float64 weights of packed codes."""
    n = wq.shape[0]
    sh = torch.arange(0, 32, bits, device=DEV, dtype=torch.int32)
    q = ((wq[..., None] >> sh) & (2**bits - 1)).view(n, -1, gs).to(F64)
    return (q * s.to(F64)[..., None] + b.to(F64)[..., None]).view(n, -1)


def _shapes(c):
    h, i, kv = c["hidden"], c["inter"], c["kv"]
    return {"q": (h, h), "k": (kv, h), "v": (kv, h), "o": (h, h), "gate": (i, h), "up": (i, h), "down": (h, i)}


def _layer_inputs(c, seed):
    """A layer's packed projections and the activations each reads."""
    g = _gen(seed)
    w = {p: _qlinear(g, n, k, c["gs"], c["bits"]) for p, (n, k) in _shapes(c).items()}
    att, o, mlp = (_randn(g, c["m"], c["hidden"]).to(BF16) for _ in range(3))
    down = _randn(g, c["m"], c["inter"]).to(BF16)
    return w, {"q": att, "k": att, "v": att, "o": o, "gate": mlp, "up": mlp, "down": down}


def _linear_inputs(c, seed):
    g = _gen(seed)
    w = _qlinear(g, c["n"], c["k"], c["gs"], c["bits"])
    x = _randn(g, c["m"], c["k"]).to(BF16)
    bias = _randn(g, c["n"]).to(BF16) if c["bias"] else None
    return w, x, bias


# ---- GGUF blocks: seeded N(0, 0.02) weights rounded to each format's grid.
# Each maker returns (block bytes uint8 [blocks, size], values float64).
_IQ4 = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)


def _u8(t):
    return t.to(torch.uint8)


def _f16b(d):
    return d.to(torch.float16).contiguous().view(torch.uint8).view(d.shape[0], 2)


def _nonzero(d):
    return torch.where(d == 0, torch.full_like(d, 1e-6), d)


def _iq4_nearest(t):
    cb = torch.tensor(_IQ4, device=DEV, dtype=F32)
    return torch.bucketize(t, (cb[1:] + cb[:-1]) / 2), cb


def _scales12(sc, m):
    """The 12-byte packing of eight 6-bit scales and mins (Q4_K, Q5_K)."""
    a = (sc[:, :4] & 63) | ((sc[:, 4:] >> 4) << 6)
    b = (m[:, :4] & 63) | ((m[:, 4:] >> 4) << 6)
    return torch.cat([a, b, (sc[:, 4:] & 15) | ((m[:, 4:] & 15) << 4)], 1)


def _asym(w, sub, levels, top):
    """Sub-block (scale, min) integers and codes of an asymmetric k-quant."""
    t = w.view(w.shape[0], -1, sub)
    lo, hi = t.amin(2).clamp(max=0), t.amax(2)
    scale, mins = (hi - lo) / (levels - 1), -lo
    d = _nonzero((scale.amax(1) / top).to(torch.float16).float())
    dm = _nonzero((mins.amax(1) / top).to(torch.float16).float())
    sc = (scale / d[:, None]).round().clamp(1, top).to(torch.int32)
    m = (mins / dm[:, None]).round().clamp(0, top).to(torch.int32)
    a, z = d[:, None] * sc, dm[:, None] * m
    q = ((t + z[..., None]) / a[..., None]).round().clamp(0, levels - 1).to(torch.int32)
    v = (d.double()[:, None] * sc)[..., None] * q - (dm.double()[:, None] * m)[..., None]
    return d, dm, sc, m, q.view(w.shape), v.view(w.shape)


def _sym(w, sub, half, top):
    """Sub-block scale integers and signed codes of a symmetric k-quant."""
    t = w.view(w.shape[0], -1, sub)
    scale = t.abs().amax(2) / half
    d = _nonzero((scale.amax(1) / top).to(torch.float16).float())
    sc = (scale / d[:, None]).round().clamp(1, top).to(torch.int32)
    q = (t / (d[:, None] * sc)[..., None]).round().clamp(-half, half - 1).to(torch.int32)
    v = (d.double()[:, None] * sc)[..., None] * q
    return d, sc, q.view(w.shape), v.view(w.shape)


def _legacy(w, half):
    d = _nonzero((w.abs().amax(1) / half).to(torch.float16).float())
    q = (w / d[:, None]).round().clamp(-half, half - 1).to(torch.int32)
    return d, q, d.double()[:, None] * q


def _q4_0(w):
    d, q, v = _legacy(w, 8)
    u = q + 8
    return torch.cat([_f16b(d), _u8(u[:, :16] | (u[:, 16:] << 4))], 1), v


def _q5_0(w):
    d, q, v = _legacy(w, 16)
    u = q + 16
    bits = ((u >> 4).view(-1, 4, 8) << torch.arange(8, device=DEV, dtype=torch.int32)).sum(2)
    return torch.cat([_f16b(d), _u8(bits), _u8((u[:, :16] & 15) | ((u[:, 16:] & 15) << 4))], 1), v


def _q8_0(w):
    d, q, v = _legacy(w, 128)
    return torch.cat([_f16b(d), q.to(torch.int8).view(torch.uint8)], 1), v


def _q2_k(w):
    d, dm, sc, m, q, v = _asym(w, 16, 4, 15)
    t = q.view(-1, 2, 4, 32)
    qs = t[:, :, 0] | (t[:, :, 1] << 2) | (t[:, :, 2] << 4) | (t[:, :, 3] << 6)
    return torch.cat([_u8(sc | (m << 4)), _u8(qs.reshape(-1, 64)), _f16b(d), _f16b(dm)], 1), v


def _q3_k(w):
    d, sc, q, v = _sym(w, 16, 4, 31)
    u = (q + 4).view(-1, 2, 4, 32)
    low, high = u & 3, u >> 2
    qs = low[:, :, 0] | (low[:, :, 1] << 2) | (low[:, :, 2] << 4) | (low[:, :, 3] << 6)
    hm = (high.view(-1, 8, 32) << torch.arange(8, device=DEV, dtype=torch.int32)[:, None]).sum(1)
    ls = sc + 32
    lo = torch.cat([(ls[:, 0:4] & 15) | ((ls[:, 8:12] & 15) << 4), (ls[:, 4:8] & 15) | ((ls[:, 12:16] & 15) << 4)], 1)
    hi = (ls[:, 0:4] >> 4) | ((ls[:, 4:8] >> 4) << 2) | ((ls[:, 8:12] >> 4) << 4) | ((ls[:, 12:16] >> 4) << 6)
    return torch.cat([_u8(hm), _u8(qs.reshape(-1, 64)), _u8(lo), _u8(hi), _f16b(d)], 1), v


def _q4_k(w):
    d, dm, sc, m, q, v = _asym(w, 32, 16, 63)
    t = q.view(-1, 4, 2, 32)
    qs = (t[:, :, 0] | (t[:, :, 1] << 4)).reshape(-1, 128)
    return torch.cat([_f16b(d), _f16b(dm), _u8(_scales12(sc, m)), _u8(qs)], 1), v


def _q5_k(w):
    d, dm, sc, m, q, v = _asym(w, 32, 32, 63)
    t = (q & 15).view(-1, 4, 2, 32)
    qs = (t[:, :, 0] | (t[:, :, 1] << 4)).reshape(-1, 128)
    qh = ((q >> 4).view(-1, 8, 32) << torch.arange(8, device=DEV, dtype=torch.int32)[:, None]).sum(1)
    return torch.cat([_f16b(d), _f16b(dm), _u8(_scales12(sc, m)), _u8(qh), _u8(qs)], 1), v


def _q6_k(w):
    d, sc, q, v = _sym(w, 16, 32, 127)
    u = (q + 32).view(-1, 2, 4, 32)
    lo, hi = u & 15, u >> 4
    ql = torch.cat([lo[:, :, 0] | (lo[:, :, 2] << 4), lo[:, :, 1] | (lo[:, :, 3] << 4)], 2)
    qh = hi[:, :, 0] | (hi[:, :, 1] << 2) | (hi[:, :, 2] << 4) | (hi[:, :, 3] << 6)
    return torch.cat([_u8(ql.reshape(-1, 128)), _u8(qh.reshape(-1, 64)), _u8(sc), _f16b(d)], 1), v


def _iq4_nl(w):
    d = _nonzero((w.abs().amax(1) / 127).to(torch.float16).float())
    q, cb = _iq4_nearest(w / d[:, None])
    v = d.double()[:, None] * cb.double()[q]
    q = q.to(torch.int32)
    return torch.cat([_f16b(d), _u8(q[:, :16] | (q[:, 16:] << 4))], 1), v


def _iq4_xs(w):
    t = w.view(-1, 8, 32)
    scale = t.abs().amax(2) / 127
    d = _nonzero((scale.amax(1) / 31).to(torch.float16).float())
    sc = (scale / d[:, None]).round().clamp(1, 31).to(torch.int32)
    q, cb = _iq4_nearest(t / (d[:, None] * sc)[..., None])
    v = ((d.double()[:, None] * sc)[..., None] * cb.double()[q]).view(w.shape)
    ls = sc + 32
    sh = ((ls >> 4) << torch.arange(0, 16, 2, device=DEV, dtype=torch.int32)).sum(1)
    sl = (ls[:, 0::2] & 15) | ((ls[:, 1::2] & 15) << 4)
    q = q.to(torch.int32)
    qs = (q[..., :16] | (q[..., 16:] << 4)).reshape(-1, 128)
    return torch.cat([_f16b(d), _u8(torch.stack([sh & 255, sh >> 8], 1)), _u8(sl), _u8(qs)], 1), v


_MAKERS = {"Q4_0": (32, _q4_0), "Q5_0": (32, _q5_0), "Q8_0": (32, _q8_0), "IQ4_NL": (32, _iq4_nl),
           "Q2_K": (256, _q2_k), "Q3_K": (256, _q3_k), "Q4_K": (256, _q4_k), "Q5_K": (256, _q5_k),
           "Q6_K": (256, _q6_k), "IQ4_XS": (256, _iq4_xs)}


def _gguf_tensor(g, kind, n, k, values):
    w = _randn(g, n, k).mul_(0.02)
    if kind in ("F16", "BF16"):
        t = w.to(torch.float16 if kind == "F16" else BF16)
        return t.view(torch.uint8).view(-1), t.double() if values else None
    e, make = _MAKERS[kind]
    data, v = make(w.view(-1, e))
    return data.reshape(-1), v.view(n, k) if values else None


def _gguf_types(c):
    return {p: c["down"] if p in ("v", "down") else c["main"] for p in PROJ}


def _gguf_inputs(c, seed, values=False):
    g, types = _gen(seed), _gguf_types(c)
    return {p: _gguf_tensor(g, types[p], n, k, values) for p, (n, k) in _shapes(c).items()}


def _heads(c, p):
    """Head count of the q/k row un-permute a conversion applies (0: none)."""
    return {"q": c["hidden"] // HEAD, "k": c["kv"] // HEAD}.get(p, 0)


def _stack_config(c):
    return stack.StackConfig(layers=c["layers"], hidden=c["hidden"], intermediate=c["inter"],
                             heads=c["hidden"] // HEAD, kv_heads=c["kv"] // HEAD, head_dim=HEAD, vocab=c["vocab"],
                             group_size=c["gs"], bits=c["bits"])


def _stack_weights(c, seed):
    """(layers of {projection: packed, ln1, ln2}, final norm, lm_head, x)."""
    g = _gen(seed)

    def norm():
        return (1 + 0.1 * _randn(g, c["hidden"])).to(BF16)

    layers = []
    for _ in range(c["layers"]):
        L = {p: _qlinear(g, n, k, c["gs"], c["bits"]) for p, (n, k) in _shapes(c).items()}
        layers.append(dict(L, ln1=norm(), ln2=norm()))
    head = _qlinear(g, c["vocab"], c["hidden"], c["gs"], c["bits"])
    return layers, norm(), head, _randn(g, c["m"], c["hidden"]).to(BF16)


# ------------------------------------------------------------------ cases
def _captured(calls):
    """A graph of the pre-bound calls, as a decode loop captures them once."""
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        for f in calls:
            f()
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        for f in calls:
            f()
    return graph


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "linear":
        w, x, bias = _linear_inputs(c, seed)
        return {"case": c, "w": w, "x": x, "bias": bias}
    if kind == "layer":
        w, x = _layer_inputs(c, seed)
        calls = [mlxq.bind_qmatmul(x[p], *w[p], c["gs"], c["bits"]) for p in PROJ]
        return {"case": c, "w": w, "x": x, "graph": _captured(calls), "out": {p: f.out for p, f in zip(PROJ, calls)},
                "calls": calls}
    if kind == "prefill":
        w, x = _layer_inputs(c, seed)
        return {"case": c, "w": w, "x": x}
    if kind == "quantize":
        w = _randn(_gen(seed), c["rows"], c["cols"]).mul_(0.02)
        return {"case": c, "w": w.to(BF16) if c["dtype"] == "bf16" else w}
    if kind == "dequantize":
        wq, s, b = _qlinear(_gen(seed), c["rows"], c["cols"], c["gs"], c["bits"])
        return {"case": c, "w": (wq, s, b) if c["dtype"] == "bf16" else (wq, s.float(), b.float())}
    if kind in ("gguf_dequant", "gguf_convert"):
        return {"case": c, "data": {p: d for p, (d, _) in _gguf_inputs(c, seed).items()}}
    layers, norm, head, x = _stack_weights(c, seed)
    st = stack.DecodeStack(_stack_config(c), batch=c["m"])
    for L, src in zip(st.layers, layers):
        for p in PROJ:
            for t, v in zip((L.proj[p].wq, L.proj[p].scales, L.proj[p].biases), src[p]):
                t.copy_(v)
        L.ln1.copy_(src["ln1"])
        L.ln2.copy_(src["ln2"])
    for t, v in zip((st.lm_head.wq, st.lm_head.scales, st.lm_head.biases), head):
        t.copy_(v)
    st.norm.copy_(norm)
    st.x.copy_(x)
    return {"case": c, "stack": st, "graph": st.capture(c["m"])}


def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "linear":
        return mlxq.qmatmul(state["x"], *state["w"], c["gs"], c["bits"], bias=state["bias"])
    if kind == "layer":
        state["graph"].replay()
        return state["out"]
    if kind == "prefill":
        w, x = state["w"], state["x"]
        return {p: mlxq.qmatmul(x[p], *w[p], c["gs"], c["bits"]) for p in PROJ}
    if kind == "quantize":
        return mlxq.quantize(state["w"], c["gs"], c["bits"])
    if kind == "dequantize":
        return mlxq.dequantize(*state["w"], c["gs"], c["bits"])
    if kind == "gguf_dequant":
        types, shapes = _gguf_types(c), _shapes(c)
        dt = BF16 if c["dtype"] == "bf16" else F32
        return {p: mlxq.gguf_dequantize(mlxq.GGUF_TAGS[types[p]], d, shapes[p][0] * shapes[p][1], dt)
                for p, d in state["data"].items()}
    if kind == "gguf_convert":
        types, shapes = _gguf_types(c), _shapes(c)
        return {p: mlxq.gguf_requantize(mlxq.GGUF_TAGS[types[p]], d, *shapes[p], _heads(c, p), c["gs"], c["bits"])
                for p, d in state["data"].items()}
    state["graph"].replay()
    return state["stack"].logits[: c["m"]]


def _packed_bytes(n, k, gs, bits):
    return n * k * bits // 8 + 4 * n * (k // gs)


def work(case):
    c, kind = case, case["kind"]
    if kind == "linear":
        b = _packed_bytes(c["n"], c["k"], c["gs"], c["bits"]) + 2 * c["m"] * (c["n"] + c["k"]) + 2 * c["n"] * c["bias"]
        return {"bytes": b, "flops": 2 * c["m"] * c["n"] * c["k"]}
    if kind in ("layer", "prefill"):
        sh = _shapes(c).values()
        b = sum(_packed_bytes(n, k, c["gs"], c["bits"]) + 2 * c["m"] * n for n, k in sh)
        b += 2 * c["m"] * (3 * c["hidden"] + c["inter"])
        return {"bytes": b, "flops": 2 * c["m"] * sum(n * k for n, k in sh)}
    if kind in ("quantize", "dequantize"):
        n, k, e = c["rows"], c["cols"], 2 if c["dtype"] == "bf16" else 4
        return {"bytes": n * k * e + n * k * c["bits"] // 8 + 2 * e * n * (k // c["gs"]), "flops": 4 * n * k}
    if kind in ("gguf_dequant", "gguf_convert"):
        types, b, f = _gguf_types(c), 0, 0
        for p, (n, k) in _shapes(c).items():
            b += mlxq.gguf_tensor_byte_len(mlxq.GGUF_TAGS[types[p]], n * k)
            if kind == "gguf_dequant":
                b += n * k * (2 if c["dtype"] == "bf16" else 4)
            else:
                b += _packed_bytes(n, k, c["gs"], c["bits"])
            f += 2 * n * k
        return {"bytes": b, "flops": f}
    sh = list(_shapes(c).values()) * c["layers"] + [(c["vocab"], c["hidden"])]
    return {"bytes": sum(_packed_bytes(n, k, c["gs"], c["bits"]) for n, k in sh) + 2 * c["m"] * (c["hidden"] + c["vocab"]),
            "flops": 2 * c["m"] * sum(n * k for n, k in sh)}


def tolerance(case):
    # codes, scales and decoded blocks are defined bit for bit
    if case["kind"] in ("quantize", "dequantize", "gguf_dequant", "gguf_convert"):
        return "exact"
    # four times what a run is from float64: a projection's bf16 output (1.7e-3)
    # plus, in the prefill kernels, weights rounded to bf16 (2.4e-3 together)
    if case["kind"] != "step":
        return {"rel": 0.01, "max": 0.06}
    return {"rel": 0.03, "max": 0.2}


def _rms64(x, w, eps=1e-5):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _affine64(w, gs, bits):
    """[None, scales, biases] of quantize in float64 (the grid's zero point is
    chosen in f32: that choice is part of the rule)."""
    edge, q0, scale = _group_params(w, gs, bits)
    s = torch.where(q0 != 0, edge.double() / torch.where(q0 != 0, q0, torch.ones_like(q0)).double(), scale.double())
    return [None, s, torch.where(q0 != 0, edge, torch.zeros_like(edge)).double()]


def _unpermute(w, heads):
    """llama.cpp's interleaved q/k rows back to half-split order."""
    if not heads:
        return w
    n, k = w.shape
    return w.view(heads, n // heads // 2, 2, k).transpose(1, 2).reshape(n, k)


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "linear":
        w, x, bias = _linear_inputs(c, seed)
        y = x.double() @ _dense64(*w, c["gs"], c["bits"]).t()
        return y if bias is None else y + bias.double()
    if kind in ("layer", "prefill"):
        w, x = _layer_inputs(c, seed)
        return {p: x[p].double() @ _dense64(*w[p], c["gs"], c["bits"]).t() for p in PROJ}
    if kind == "quantize":
        return _affine64(prepare(c, seed)["w"], c["gs"], c["bits"])
    if kind == "dequantize":
        return _dense64(*prepare(c, seed)["w"], c["gs"], c["bits"])
    if kind == "gguf_dequant":
        return {p: v.reshape(-1) for p, (_, v) in _gguf_inputs(c, seed, True).items()}
    if kind == "gguf_convert":
        return {p: _affine64(_unpermute(v.float().to(BF16), _heads(c, p)), c["gs"], c["bits"])
                for p, (_, v) in _gguf_inputs(c, seed, True).items()}
    layers, norm, head, x = _stack_weights(c, seed)
    dense = lambda t: _dense64(*t, c["gs"], c["bits"]).t()  # noqa: E731
    x = x.double()
    for L in layers:
        v = _rms64(x, L["ln1"]) @ dense(L["v"])
        v = v.view(c["m"], -1, 1, HEAD).expand(-1, -1, c["hidden"] // c["kv"], -1).reshape(c["m"], -1)
        h = x + v @ dense(L["o"])
        n = _rms64(h, L["ln2"])
        a = torch.nn.functional.silu(n @ dense(L["gate"])) * (n @ dense(L["up"]))
        x = h + a @ dense(L["down"])
    n = _rms64(x, norm)
    # the head in row blocks: its float64 weights would take gigabytes
    wq, s, b = head
    return torch.cat([n @ dense((wq[r:r + 8192], s[r:r + 8192], b[r:r + 8192])) for r in range(0, c["vocab"], 8192)], 1)
