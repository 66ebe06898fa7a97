"""Performance cases of the Q4_K library: what a user of it has it do, through
its public entry points (modgrad_amd.q4k, modgrad_amd.arena).

A case is a dict of plain values; "kind" names the path:

  linear   LinearResidentQuantized.forward: flattened Q4_K weight, bias
  layer    the seven matvecs of a decoder layer, launched one by one
  chain    a whole decode step's matvecs as one recorded chain
  ops      a decode step's layers with their norms, GLU and residuals, in the
           Q4_K / Q6_K mix of a Q4_K_M file, recorded as one op chain
  dp4a     a layer on Q8_1 activations (quantize + int8 matvec)
  kquant   a layer of Q5_K and Q6_K tensors from a weight arena
  batched  multi-sequence decode: one layer's FFN matrices, 2 to 16 rows of X
  prefill  the four GEMMs of a decoder layer over `tokens` prompt tokens
  dequant  Q4_K -> f32 of a resident tensor

Weights are synthetic blocks whose values are spread as those of a quantized
N(0, 0.02) matrix; activations are N(0, 1).
"""
from __future__ import annotations

import math

import torch

from modgrad_amd import _lib
from modgrad_amd.arena import WeightArena
from modgrad_amd.gguf import GgmlType
from modgrad_amd.q4k import (Chain, GpuVec, LinearResidentQuantized, kern, op_matvec,
                             op_matvec_glu, op_matvec_norm, op_residual_add, ops)

EPS = 1e-6


# ------------------------------------------------------------------- cases --

def listed():
    layer7b = {"hidden": 3584, "inter": 18944, "kv": 512}
    return [
        # the smallest call: one quantized linear layer of a 0.5B-class model
        # (its rows are no whole blocks, so the flattened layout)
        {"name": "linear_4864x896", "kind": "linear", "out": 4864, "in": 896},
        # the calling pattern of an engine that launches every matvec itself:
        # launch latency and short kernels (k, v) beside streaming ones
        {"name": "layer_7b_eager", "kind": "layer", **layer7b},
        # the headline: one token of a 7B-class model, 113 matvecs, one graph
        {"name": "decode_7b_chain", "kind": "chain", **layer7b, "layers": 28, "vocab": 152064},
        # a Q4_K_M file's decode step with its glue fused, four layers and the head
        {"name": "decode_q4km_ops", "kind": "ops", **layer7b, "layers": 4, "vocab": 152064},
        # the int8-activation arm, the default of the engine this library serves
        {"name": "layer_7b_dp4a", "kind": "dp4a", **layer7b},
        # a Q5_K_M file's layer: Q5_K with v and down in Q6_K
        {"name": "layer_7b_q5km", "kind": "kquant", **layer7b, "align": 256},
        # eight sequences decoded together
        {"name": "ffn_batched_8", "kind": "batched", "hidden": 3584, "inter": 18944, "batch": 8},
        # a short prompt, or the draft of a speculative step: few, ragged tokens
        {"name": "prefill_45", "kind": "prefill", **layer7b, "tokens": 45},
        # a chunk of a scheduler that mixes prefill with decode
        {"name": "prefill_160", "kind": "prefill", **layer7b, "tokens": 160},
        # an ordinary prompt
        {"name": "prefill_512", "kind": "prefill", **layer7b, "tokens": 512},
        # a long prompt, the largest case
        {"name": "prefill_4096", "kind": "prefill", **layer7b, "tokens": 4096},
        # the f32 copy that a dequantizing caller (training, export) asks for
        {"name": "dequant_18944x3584", "kind": "dequant", "blocks": 18944 * 14},
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, even over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _layer_dims(rng):
    """Layer sizes from a 1B-class to a 14B-class model; kv is 1/8 to 1/1 of
    hidden, row counts odd now and then (pruned or sharded matrices)."""
    hidden = 256 * rng.randint(6, 20)
    inter = 256 * max(8, int(hidden * rng.uniform(2.5, 5.3)) // 256)
    return {"hidden": hidden, "inter": inter, "kv": 64 * rng.randint(2, hidden // 64)}


def draw(rng):
    kind = rng.choice(["linear", "layer", "chain", "ops", "dp4a", "kquant", "batched", "prefill",
                       "prefill", "prefill", "dequant"])
    if kind == "linear":
        k = 32 * _log(rng, 8, 128)
        n = _log(rng, 64, 16384)
        while n * k % 256:
            n += 1
        return {"kind": kind, "out": n, "in": k}
    if kind == "batched":
        d = _layer_dims(rng)
        return {"kind": kind, "hidden": d["hidden"], "inter": d["inter"], "batch": rng.randint(2, 16)}
    if kind == "dequant":
        return {"kind": kind, "blocks": _log(rng, 1000, 400000)}
    case = {"kind": kind, **_layer_dims(rng)}
    if kind == "chain":
        case.update(layers=_log(rng, 2, 24), vocab=_log(rng, 16000, 152064))
    elif kind == "ops":
        # the fused norm before a Q6_K tensor takes rows of up to 14 blocks
        case["hidden"] = min(case["hidden"], 3584)
        case["kv"] = min(case["kv"], case["hidden"])
        case.update(layers=_log(rng, 1, 8), vocab=8 * _log(rng, 2000, 19008))
    elif kind == "kquant":
        case["align"] = rng.choice([256, 256, 256, 2])
    elif kind == "prefill":
        # no more than the largest listed case's work
        most = 4096 * _prefill_weights({"hidden": 3584, "inter": 18944, "kv": 512})
        case["tokens"] = min(_log(rng, 17, 4096), most // _prefill_weights(case))
    return case


# ----------------------------------------------------- synthetic quantities --

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _bytes(g, *shape):
    return torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=g)


def _scales(g, nblk):
    """The 16 header bytes of Q4_K and Q5_K blocks: f16 d and dmin, 8 six-bit
    scales and 8 six-bit mins, the mins near the scales so that the weights
    are centred, as a quantizer leaves them."""
    r = torch.randint(0, 32, (2, nblk, 8), dtype=torch.uint8, device="cuda", generator=g)
    sc = r[0] + 32
    mn = (sc + (r[1] >> 2)).sub_(4).clamp_(max=63)
    out = torch.empty((nblk, 16), dtype=torch.uint8, device="cuda")
    d = torch.rand((nblk, 1), device="cuda", generator=g) * 1.2e-4 + 7e-5
    return out, sc, mn, d


def _pack_header(out, sc, mn, d, centre):
    out[:, 0:4] = torch.cat([d, d * centre], 1).to(torch.float16).view(torch.uint8)
    lo, hi = slice(0, 4), slice(4, 8)
    out[:, 4:8] = sc[:, lo] | ((sc[:, hi] >> 4) << 6)
    out[:, 8:12] = mn[:, lo] | ((mn[:, hi] >> 4) << 6)
    out[:, 12:16] = (sc[:, hi] & 15) | ((mn[:, hi] & 15) << 4)


def _nibbles(g, nblk, n):
    """n bytes of two 4-bit values each, every value the mean of two uniform
    ones (a hump around 7, as quantized normal weights have)."""
    a, b = _bytes(g, nblk, n), _bytes(g, nblk, n)
    hi = ((a >> 4) + (b >> 4)) >> 1
    return ((a & 15).add_(b & 15) >> 1).bitwise_or_(hi << 4)


_CHUNK = 1 << 20  # blocks made at a time


def _weight(dtype, n, k, g):
    """The bytes of an n x k weight of the given GGML type."""
    nblk = n * k // 256
    size = {GgmlType.Q4_K: 144, GgmlType.Q5_K: 176, GgmlType.Q6_K: 210}[dtype]
    w = torch.empty((nblk, size), dtype=torch.uint8, device="cuda")
    for b0 in range(0, nblk, _CHUNK):
        m = min(_CHUNK, nblk - b0)
        part = w[b0:b0 + m]
        if dtype == GgmlType.Q6_K:
            part[:, :128] = _nibbles(g, m, 128)
            part[:, 128:192] = _bytes(g, m, 64)
            part[:, 192:208] = _bytes(g, m, 16) // 4 + 40
            d = torch.rand((m, 1), device="cuda", generator=g) * 1.2e-5 + 7e-6
            part[:, 208:210] = d.to(torch.float16).view(torch.uint8)
            continue
        head, sc, mn, d = _scales(g, m)
        if dtype == GgmlType.Q5_K:
            _pack_header(head, sc, mn, d * 0.5, 15.0)
            part[:, 16:48] = _bytes(g, m, 32)
        else:
            _pack_header(head, sc, mn, d, 7.0)
        part[:, :16] = head
        part[:, -128:] = _nibbles(g, m, 128)
    return w.view(-1)


def _randn(g, *shape, dtype=torch.float32):
    return torch.randn(shape, device="cuda", generator=g).to(dtype)


def _dequant(dtype, w, f64=True):
    """Blocks of bytes -> [blocks, 256] weights in 64 bits, by the format."""
    t = torch.float64 if f64 else torch.float32
    if dtype == GgmlType.Q6_K:
        b = w.view(-1, 210)
        ql, qh = b[:, :128].view(-1, 2, 2, 32), b[:, 128:192].view(-1, 2, 1, 32)
        low = torch.cat([ql & 15, ql >> 4], 2)  # 128-half, quarter, position
        shift = torch.tensor([0, 2, 4, 6], dtype=torch.uint8, device=w.device).view(1, 1, 4, 1)
        q = (low | (((qh >> shift) & 3) << 4)).to(t) - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).to(t).view(-1, 2, 4, 2, 1)
        d = b[:, 208:210].contiguous().view(torch.float16).to(t).view(-1, 1, 1, 1, 1)
        return (d * sc * q.view(-1, 2, 4, 2, 16)).view(-1, 256)
    b = w.view(-1, 144 if dtype == GgmlType.Q4_K else 176)
    dd = b[:, :4].contiguous().view(torch.float16).to(t)
    s = b[:, 4:16]
    sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1)
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
    qs = b[:, -128:].reshape(-1, 4, 1, 32)
    q = torch.cat([qs & 15, qs >> 4], 2).view(-1, 8, 32)
    if dtype == GgmlType.Q5_K:
        bit = torch.arange(8, dtype=torch.uint8, device=w.device).view(1, 8, 1)
        q = q | (((b[:, 16:48].reshape(-1, 1, 32) >> bit) & 1) << 4)
    scale = (dd[:, :1] * sc.to(t)).unsqueeze(2)
    return (scale * q.to(t) - (dd[:, 1:] * mn.to(t)).unsqueeze(2)).view(-1, 256)


def _matmul64(dtype, w, n, k, x):
    """x @ W^T in 64 bits, [rows, n] (or [n] for one vector), by row ranges."""
    x = x.to(torch.float64)
    rows = max(1, (1 << 27) // k)
    rows += -rows * k % 256
    while rows * k % 256:
        rows += 1
    out = []
    wb = w.view(-1)
    bb = {GgmlType.Q4_K: 144, GgmlType.Q5_K: 176, GgmlType.Q6_K: 210}[dtype]
    for r0 in range(0, n, rows):
        r1 = min(n, r0 + rows)
        m = _dequant(dtype, wb[r0 * k // 256 * bb: r1 * k // 256 * bb]).view(r1 - r0, k)
        out.append(x @ m.t() if x.dim() == 2 else m @ x)
    return torch.cat(out, -1)


def _round16(n):
    return -(-n // 16) * 16


def _slots(sizes, dtype=torch.float32):
    """One buffer, and each part of it (parts start 64 bytes apart at least)."""
    buf = torch.zeros(sum(_round16(s) for s in sizes), dtype=dtype, device="cuda")
    parts, at = [], 0
    for s in sizes:
        parts.append(buf[at:at + s])
        at += _round16(s)
    return buf, parts


# ---------------------------------------------------------------- per kind --

def _layer_shapes(c):
    h, i, kv = c["hidden"], c["inter"], c["kv"]
    return [("q", h, h), ("k", kv, h), ("v", kv, h), ("o", h, h), ("gate", i, h), ("up", i, h),
            ("down", h, i)]


def _fused_shapes(c):
    h, i, kv = c["hidden"], c["inter"], c["kv"]
    return [("qkv", h + 2 * kv, h), ("o", h, h), ("gate_up", 2 * i, h), ("down", h, i)]


def _prefill_weights(c):
    return sum(n * k for _, n, k in _fused_shapes(c))


def _chain_shapes(c):
    return _fused_shapes(c) * c["layers"] + [("lm_head", c["vocab"], c["hidden"])]


def _dtype_of(kind, name, layer=0):
    if kind == "ops":
        # 'more bits' tensors of a Q4_K_M file: v and down on every other layer
        return GgmlType.Q6_K if name in ("v", "down") and layer % 2 == 0 else GgmlType.Q4_K
    if kind == "kquant":
        return GgmlType.Q6_K if name in ("v", "down") else GgmlType.Q5_K
    if kind == "dp4a":
        return GgmlType.Q6_K if name == "down" else GgmlType.Q4_K
    return GgmlType.Q4_K


def _arena(items, align):
    """A weight arena holding the given (name, dims, type, device bytes)."""
    a = WeightArena([(n, d, t) for n, d, t, _ in items], align)
    for n, _, _, data in items:
        a.tensor(n).copy_(data.view(torch.uint8).view(-1))
    return a


def prepare(case, seed):
    c, g = case, _gen(seed)
    kind = c["kind"]
    s = {"case": c}
    if kind == "linear":
        w = _weight(GgmlType.Q4_K, c["out"], c["in"], g)
        lin = LinearResidentQuantized.from_q4k(w.cpu().numpy(), _randn(g, c["out"]).cpu().numpy(),
                                               c["in"], c["out"])
        lin.ensure_resident()
        x, y = GpuVec.try_hip(c["in"]), GpuVec.try_hip(c["out"])
        x.copy_from(_randn(g, c["in"]).cpu().numpy())
        s.update(lin=lin, x=x, y=y, out=y.hip_buffer().tensor().view(torch.float32))
    elif kind in ("layer", "chain"):
        shapes = _layer_shapes(c) if kind == "layer" else _chain_shapes(c)
        s["out"], ys = _slots([n for _, n, _ in shapes])
        s["jobs"] = [(_weight(GgmlType.Q4_K, n, k, g), _randn(g, k), y, n, k // 256)
                     for (_, n, k), y in zip(shapes, ys)]
        if kind == "chain":
            s["chain"] = Chain([(w.data_ptr(), x.data_ptr(), y.data_ptr(), n, b)
                                for w, x, y, n, b in s["jobs"]])
    elif kind == "ops":
        _prepare_ops(c, g, s)
    elif kind in ("dp4a", "kquant"):
        shapes = _layer_shapes(c)
        items = [(nm, [k, n], _dtype_of(kind, nm), _weight(_dtype_of(kind, nm), n, k, g))
                 for nm, n, k in shapes]
        s["arena"] = _arena(items, c.get("align", 256))
        s["out"], ys = _slots([n for _, n, _ in shapes])
        s["jobs"] = [(nm, _randn(g, k), y, n, k) for (nm, n, k), y in zip(shapes, ys)]
        if kind == "dp4a":
            km = max(k for _, _, k in shapes)
            s["q8"] = (torch.zeros(km, dtype=torch.int8, device="cuda"),
                       torch.zeros(km // 32, device="cuda"), torch.zeros(km // 32, device="cuda"))
    elif kind == "batched":
        h, i, b = c["hidden"], c["inter"], c["batch"]
        shapes = [(2 * i, h), (h, i)]
        ws = max(kern.batched_workspace_bytes(k // 256, b) for _, k in shapes)
        s["workspace"] = torch.empty(ws, dtype=torch.uint8, device="cuda")
        s["jobs"] = [(_weight(GgmlType.Q4_K, n, k, g), _randn(g, b, k),
                      torch.zeros((b, n), device="cuda"), n, k // 256) for n, k in shapes]
    elif kind == "prefill":
        m = c["tokens"]
        s["jobs"] = [(_weight(GgmlType.Q4_K, n, k, g), _randn(g, m, k, dtype=torch.float16),
                      torch.zeros((m, n), device="cuda"), n, k // 256)
                     for _, n, k in _fused_shapes(c)]
    else:
        s["w"] = _weight(GgmlType.Q4_K, c["blocks"], 256, g)
        s["out"] = torch.zeros(c["blocks"] * 256, device="cuda")
    return s


def _prepare_ops(c, g, s):
    h, i, kv = c["hidden"], c["inter"], c["kv"]
    s["emb"], s["h"] = _randn(g, h), torch.zeros(h, device="cuda")
    s["logits"] = torch.zeros(c["vocab"], device="cuda")
    s["qkv"], parts = _slots([h, kv, kv] * c["layers"])
    o, f, dn = (torch.zeros(n, device="cuda") for n in (h, i, h))
    s["layers"], chain = [], []
    for l in range(c["layers"]):
        ly = {nm: _weight(_dtype_of("ops", nm, l), n, k, g) for nm, n, k in _layer_shapes(c)}
        # what attention hands to the o projection (attention is the caller's)
        ly["attn"] = _randn(g, h)
        ly["n1"], ly["n2"] = 1 + 0.1 * _randn(g, h), 1 + 0.1 * _randn(g, h)
        s["layers"].append(ly)
        p = {nm: t.data_ptr() for nm, t in ly.items()}
        q, k, v = (t.data_ptr() for t in parts[3 * l:3 * l + 3])
        hp, op, fp, dp = (t.data_ptr() for t in (s["h"], o, f, dn))
        chain += [op_matvec_norm(p["q"], hp, p["n1"], EPS, q, h, h),
                  op_matvec_norm(p["k"], hp, p["n1"], EPS, k, kv, h),
                  op_matvec_norm(p["v"], hp, p["n1"], EPS, v, kv, h, int(_dtype_of("ops", "v", l))),
                  op_matvec(_lib.DTYPE_Q4_K, p["o"], p["attn"], op, h, h),
                  op_residual_add(hp, op, h),
                  op_matvec_glu(p["gate"], p["up"], hp, fp, i, h, p["n2"], EPS),
                  op_matvec(int(_dtype_of("ops", "down", l)), p["down"], fp, dp, h, i),
                  op_residual_add(hp, dp, h)]
    s["head"], s["n3"] = _weight(GgmlType.Q6_K, c["vocab"], h, g), 1 + 0.1 * _randn(g, h)
    chain.append(op_matvec_norm(s["head"].data_ptr(), s["h"].data_ptr(), s["n3"].data_ptr(), EPS,
                                s["logits"].data_ptr(), c["vocab"], h, _lib.DTYPE_Q6_K))
    s["scratch"] = (o, f, dn)
    s["chain"] = Chain.from_ops(chain)


def run(s):
    kind = s["case"]["kind"]
    if kind == "linear":
        s["lin"].forward(s["x"], s["y"])
        return s["out"]
    if kind == "layer":
        for w, x, y, n, b in s["jobs"]:
            kern.matvec_q4k(w.data_ptr(), x.data_ptr(), y.data_ptr(), n, b)
        return s["out"]
    if kind == "chain":
        s["chain"].launch()
        return s["out"]
    if kind == "ops":
        s["h"].copy_(s["emb"])
        s["chain"].launch()
        return {"h": s["h"], "qkv": s["qkv"], "logits": s["logits"]}
    if kind == "kquant":
        for nm, x, y, n, k in s["jobs"]:
            s["arena"].qmatvec(nm, x.data_ptr(), y.data_ptr())
        return s["out"]
    if kind == "dp4a":
        q8 = tuple(t.data_ptr() for t in s["q8"])
        for nm, x, y, n, k in s["jobs"]:
            if s["arena"].dtype[nm] == GgmlType.Q6_K:
                kern.quantize_q8_1(x.data_ptr(), *q8, k)
                kern.matvec_q6k_dp4a(s["arena"].ptr(nm), *q8, y.data_ptr(), n, k // 256)
            else:
                s["arena"].qmatvec(nm, x.data_ptr(), y.data_ptr(), q8=q8)
        return {"y": s["out"], "xq": s["q8"][0], "xd": s["q8"][1], "xsum": s["q8"][2]}
    if kind == "batched":
        for w, x, y, n, b in s["jobs"]:
            kern.matvec_q4k_batched(w.data_ptr(), x.data_ptr(), y.data_ptr(), n, b,
                                    s["case"]["batch"], workspace=s["workspace"])
        return [j[2] for j in s["jobs"]]
    if kind == "prefill":
        for w, a, y, n, b in s["jobs"]:
            kern.gemm_q4k_f16(w.data_ptr(), a.data_ptr(), y.data_ptr(), n, b, s["case"]["tokens"])
        return [j[2] for j in s["jobs"]]
    ops.dequant_q4k_resident(s["w"].data_ptr(), s["out"].data_ptr(), s["case"]["blocks"])
    return s["out"]


# ------------------------------------------------------------------- exact --

def _q8_1(x):
    """Q8_1 of x: int8 values, scale and sum per 32, in the format's 32-bit steps."""
    v = x.cpu().view(-1, 32)
    amax = v.abs().amax(1)
    inv = torch.where(amax > 0, 127.0 / amax, torch.zeros_like(amax))
    q = torch.round(v * inv[:, None]).clamp(-127, 127)
    return q.to(torch.float64).cuda(), (amax / 127.0).cuda(), q.sum(1).cuda()


def exact(case, seed):
    c = case
    kind = c["kind"]
    s = prepare(case, seed)
    if kind == "linear":
        w = torch.from_numpy(s["lin"].host_weight_q4k).cuda()
        x = s["x"].hip_buffer().tensor().view(torch.float32)
        b = torch.from_numpy(s["lin"].host_bias).cuda().to(torch.float64)
        return _matmul64(GgmlType.Q4_K, w, c["out"], c["in"], x) + b
    if kind in ("layer", "chain", "kquant", "dp4a"):
        out = torch.zeros(s["out"].numel(), dtype=torch.float64, device="cuda")
        at, last = 0, None
        for w, x, y, n, b in s["jobs"]:
            t, k = GgmlType.Q4_K, x.numel()
            if kind in ("kquant", "dp4a"):
                t, w = s["arena"].dtype[w], s["arena"].tensor(w).clone()
            if kind == "dp4a":
                q, d, sums = last = _q8_1(x)
                x = (q * d[:, None].to(torch.float64)).view(-1)
            out[at:at + n] = _matmul64(t, w, n, k, x)
            at += _round16(n)
        if kind != "dp4a":
            return out
        # the buffers hold the last job's activations, the widest or not
        xq, xd, xsum = (t.to(torch.float64).clone() for t in s["q8"])
        for _, x, _, _, k in s["jobs"]:
            q, d, sums = _q8_1(x)
            xq[:k], xd[:k // 32], xsum[:k // 32] = q.view(-1), d, sums
        return {"y": out, "xq": None, "xd": xd, "xsum": xsum}
    if kind == "ops":
        return _exact_ops(c, s)
    if kind in ("batched", "prefill"):
        return [_matmul64(GgmlType.Q4_K, w, n, b * 256, x) for w, x, _, n, b in s["jobs"]]
    return _dequant(GgmlType.Q4_K, s["w"]).view(-1)


def _exact_ops(c, s):
    h, f64 = s["emb"].to(torch.float64), torch.float64
    qkv, at = torch.zeros(s["qkv"].numel(), dtype=f64, device="cuda"), 0

    def norm(v, w):
        return v / torch.sqrt((v * v).mean() + EPS) * w.to(f64)

    for l, ly in enumerate(s["layers"]):
        y = {}
        for nm, n, k in _layer_shapes(c):
            if nm in ("q", "k", "v"):
                x = norm(h, ly["n1"])
            elif nm == "o":
                x = ly["attn"]
            elif nm in ("gate", "up"):
                x = norm(h, ly["n2"])
            else:
                x = torch.nn.functional.gelu(y["gate"], approximate="tanh") * y["up"]
            y[nm] = _matmul64(_dtype_of("ops", nm, l), ly[nm], n, k, x)
            if nm in ("q", "k", "v"):
                qkv[at:at + n] = y[nm]
                at += _round16(n)
            elif nm in ("o", "down"):
                h = h + y[nm]
    logits = _matmul64(GgmlType.Q6_K, s["head"], c["vocab"], c["hidden"], norm(h, s["n3"]))
    return {"h": h, "qkv": qkv, "logits": logits}


# --------------------------------------------------------- work, tolerance --

_BYTES = {GgmlType.Q4_K: 144, GgmlType.Q5_K: 176, GgmlType.Q6_K: 210}


def _product(n, k, rows=1, dtype=GgmlType.Q4_K, xbytes=4):
    """(bytes, flops) of rows x [n, k]: weights, activations in, results out."""
    return (n * k // 256 * _BYTES[dtype] + rows * (xbytes * k + 4 * n), 2 * rows * n * k)


def work(case):
    c = case
    kind = c["kind"]
    if kind == "linear":
        jobs = [_product(c["out"], c["in"]), (4 * c["out"], c["out"])]
    elif kind == "layer":
        jobs = [_product(n, k) for _, n, k in _layer_shapes(c)]
    elif kind == "chain":
        jobs = [_product(n, k) for _, n, k in _chain_shapes(c)]
    elif kind == "ops":
        jobs = [_product(n, k, dtype=_dtype_of(kind, nm, l))
                for l in range(c["layers"]) for nm, n, k in _layer_shapes(c)]
        jobs.append(_product(c["vocab"], c["hidden"], dtype=GgmlType.Q6_K))
    elif kind in ("dp4a", "kquant"):
        jobs = [_product(n, k, dtype=_dtype_of(kind, nm)) for nm, n, k in _layer_shapes(c)]
    elif kind == "batched":
        h, i, b = c["hidden"], c["inter"], c["batch"]
        jobs = [_product(2 * i, h, b), _product(h, i, b)]
    elif kind == "prefill":
        jobs = [_product(n, k, c["tokens"], xbytes=2) for _, n, k in _fused_shapes(c)]
    else:
        jobs = [(c["blocks"] * (144 + 1024), 2 * 256 * c["blocks"])]
    return {"bytes": sum(b for b, _ in jobs), "flops": sum(f for _, f in jobs)}


def tolerance(case):
    kind = case["kind"]
    if kind == "dequant":
        return "exact"  # the format fixes every rounding
    # about four times the error against 64 bits, over the ranges
    if kind == "prefill":
        # weights and activations are f16 matrix-core operands (7e-4)
        return {"rel": 2.8e-3, "max": 2e-2}
    if kind == "ops":
        # layers and norms in sequence, each in 32 bits (1.6e-5)
        return {"rel": 6e-5, "max": 6e-4}
    return {"rel": 2e-5, "max": 2e-4}  # 32-bit sums (up to 5e-6)
