"""Performance cases of rq: the calls a program makes against resident quantized weights.

A case is a dict of plain values; `op` names the call:

  linear     y = x . dequant(W)^T through QWeight.matmul (Q8_0, Q4_0, Q4_K, Q6_K)
  linear_i8  int8-activation prefill: quantize_act_i8, then QWeight.matmul_i8
  train      a frozen quantized linear in a training step: y forward, dx backward
  decoder    DecoderLayer.step over a stack of layers, one new token
  attention  decode_attention: RoPE, KV append and one query over a cache
  encode     a float weight to Q8_0, Q4_K or Q6_K on the device, at load time

Weights are N(0, 0.02^2) matrices quantized to the case's format (the torch
restatement of each format's encoder below), activations N(0, 1).
"""
import math

import torch

import raster_amd
from raster_amd.decoder import DecoderLayer

# the shapes come from the benchmark's configurations: 4096 x 4096, 4096 ->
# 11008, 4096 -> 14336, 8192 -> 28672, and the decoder of d 2048 / ffn 5632


def listed():
    return [
        # one token through a square projection: the smallest call, launch and latency bound
        {"name": "decode_q8_m1", "op": "linear", "fmt": "q8", "x": "f32", "y": "f32", "m": 1, "in": 4096, "out": 4096},
        # a few sequences decoding together through an FFN up projection
        {"name": "decode_q4_m4", "op": "linear", "fmt": "q4h", "x": "f32", "y": "f32", "m": 4, "in": 4096,
         "out": 14336},
        # one token against a K-quant weight, the format of most small-memory deployments
        {"name": "decode_q4k_m1", "op": "linear", "fmt": "q4k", "x": "f32", "y": "f32", "m": 1, "in": 4096,
         "out": 14336},
        # a prompt through an FFN projection, bf16 activations
        {"name": "prefill_q8_bf16", "op": "linear", "fmt": "q8", "x": "bf16", "y": "bf16", "m": 512, "in": 4096,
         "out": 11008},
        # a long prompt through the FFN of a large model: the largest call
        {"name": "prefill_q8_bf16_large", "op": "linear", "fmt": "q8", "x": "bf16", "y": "bf16", "m": 2048,
         "in": 8192, "out": 28672},
        # a ragged prompt with f32 activations, Raster's default type, and Q4_0's own f32 scales
        {"name": "prefill_q4_f32", "op": "linear", "fmt": "q4f", "x": "f32", "y": "f32", "m": 333, "in": 4096,
         "out": 11008},
        # the same prompt work against a K-quant weight
        {"name": "prefill_q6k", "op": "linear", "fmt": "q6k", "x": "f32", "y": "f32", "m": 512, "in": 4096,
         "out": 11008},
        # int8 prefill: Raster's own GPU prefill route (quantized activations, exact integer dots)
        {"name": "prefill_i8", "op": "linear_i8", "fmt": "q8", "y": "bf16", "m": 512, "in": 4096, "out": 11008},
        # a training step's frozen linear (adapters above it): forward and backward-data
        {"name": "train_q8", "op": "train", "fmt": "q8", "m": 512, "in": 2048, "out": 5632},
        # one decode step of a two-layer decoder, launched call by call
        {"name": "decoder_step", "op": "decoder", "layers": 2, "heads": 16, "kv_heads": 16, "hd": 128, "ffn": 5632,
         "cached": 128},
        # grouped-query attention of one token over a long cache
        {"name": "attention_gqa", "op": "attention", "heads": 32, "kv_heads": 8, "hd": 128, "cached": 4096},
        # a weight quantized when it is loaded; its rows are padded to whole super-blocks
        {"name": "encode_q4k", "op": "encode", "fmt": "q4k", "in": 4000, "out": 11008},
    ]


# the most work (m * in * out) a drawn linear has: bf16 x as the largest listed
# case, everything else as a 512-row prompt through 4096 -> 11008
_MOST = 512 * 4096 * 11008
_MOST_BF16 = 2048 * 8192 * 28672


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["linear"] * 6 + ["linear_i8", "train", "decoder", "attention", "encode"])
    if op == "decoder":
        heads = rng.choice([8, 12, 16, 24])
        return {"op": op, "layers": rng.choice([1, 2]), "heads": heads, "kv_heads": heads // rng.choice([1, 2, 4]),
                "hd": 128, "ffn": 32 * rng.randint(32, 200), "cached": _log(rng, 16, 1024)}
    if op == "attention":
        kv = rng.choice([2, 4, 8, 16])
        return {"op": op, "heads": kv * rng.choice([1, 2, 4, 8]), "kv_heads": kv, "hd": rng.choice([64, 128]),
                "cached": _log(rng, 32, 16384)}
    if op == "encode":
        fmt = rng.choice(["q8", "q4k", "q6k"])
        in_ = {"q8": 32, "q4k": 8, "q6k": 256}[fmt]
        in_ *= _log(rng, 1024 // in_, 8192 // in_)
        return {"op": op, "fmt": fmt, "in": in_, "out": _log(rng, 512, 8192)}
    fmt = rng.choice(["q8", "q4h", "q4f"] if op == "linear_i8" else ["q8", "q4h"] if op == "train"
                     else ["q8", "q8", "q4h", "q4f", "q4k", "q6k"])
    step = 256 if fmt in ("q4k", "q6k") else 32
    in_, out = step * _log(rng, 1024 // step, 8192 // step), _log(rng, 1024, 28672)
    y = rng.choice(["f32", "bf16"])
    if op == "linear":
        x = "f32" if step == 256 else rng.choice(["f32", "bf16"])
        most = _MOST_BF16 if x == "bf16" else _MOST
        m = min(_log(rng, 1, 2048 if x == "bf16" else 1024), most // (in_ * out))
        return {"op": op, "fmt": fmt, "x": x, "y": y, "m": m, "in": in_, "out": out}
    m = min(_log(rng, 17, 1024), _MOST // (2 * in_ * out) if op == "train" else _MOST // (in_ * out))
    case = {"op": op, "fmt": fmt, "m": m, "in": in_, "out": out}
    return case if op == "train" else {**case, "y": y}


# ---- inputs -------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _round(v, lo, hi):
    return torch.floor(v + 0.5).clamp_(lo, hi)


def _inv(d):
    return torch.where(d == 0, torch.zeros_like(d), 1.0 / d)


def _float_weight(g, out, in_):
    return torch.randn((out, in_), generator=g, device="cuda") * 0.02


def _blocks(w, n):
    return w.double().view(w.shape[0], -1, n)


def _q8(w):
    b = _blocks(w, 32)
    d = b.abs().amax(2, keepdim=True) / 127.0
    return _round(b * _inv(d), -127, 127), d.float()


def _q4(w, half):
    b = _blocks(w, 32)
    d = b.abs().amax(2, keepdim=True) / 7.0
    return _round(b * _inv(d) + 8.0, 0, 15), d.half() if half else d.float()


def _q4k(w):
    b = _blocks(w, 32).view(w.shape[0], -1, 8, 32)
    lo = b.amin(3)
    a = (b.amax(3) - lo) / 15.0
    da, db = a.amax(2, keepdim=True) / 63.0, lo.abs().amax(2, keepdim=True) / 31.0
    aq, bq = _round(a * _inv(da), 0, 63), _round(lo * _inv(db), -32, 31)
    q = _round((b - (db * bq)[..., None]) * _inv(da * aq)[..., None], 0, 15)
    return q, da.float(), db.float(), aq, bq


def _q6k(w):
    b = _blocks(w, 16).view(w.shape[0], -1, 16, 16)
    a = b.abs().amax(3) / 32.0
    d = a.amax(2, keepdim=True) / 127.0
    sc = _round(a * _inv(d), 0, 127)
    return _round(b * _inv(d * sc)[..., None], -32, 31) + 32, sc, d.float()


def _nibbles(q):
    """Codes [..., 32] to bytes: element k low, element k + 16 high."""
    q = q.to(torch.uint8)
    return (q[..., :16] | (q[..., 16:] << 4)).cpu().numpy().ravel()


def _host(t, dtype=None):
    return (t if dtype is None else t.to(dtype)).cpu().numpy().ravel()


def _weight(fmt, w):
    """The float weight w [out, in] as a resident weight of the format."""
    out, in_ = w.shape
    ctx = raster_amd.context(0)
    if fmt == "q8":
        q, d = _q8(w)
        return raster_amd.QWeight.q8(_host(q, torch.int8), _host(d), out, in_, ctx)
    if fmt in ("q4h", "q4f"):
        q, d = _q4(w, fmt == "q4h")
        return raster_amd.QWeight.q4(_nibbles(q), _host(d), out, in_, ctx)
    if fmt == "q4k":
        q, da, db, aq, bq = _q4k(w)
        return raster_amd.QWeight.q4k(_nibbles(q), _host(da), _host(db), _host(aq, torch.uint8), _host(bq, torch.int8),
                                      out, in_, ctx)
    q, sc, d = _q6k(w)
    return raster_amd.QWeight.q6k(_host(q, torch.uint8), _host(sc, torch.int8), _host(d), out, in_, ctx)


def _dense(fmt, w):
    """The weight's dequantized values in 64 bits, [out, in]."""
    if fmt == "q8":
        q, d = _q8(w)
        v = q * d.double()
    elif fmt in ("q4h", "q4f"):
        q, d = _q4(w, fmt == "q4h")
        v = (q - 8.0) * d.double()
    elif fmt == "q4k":
        q, da, db, aq, bq = _q4k(w)
        v = q * (da.double() * aq)[..., None] + (db.double() * bq)[..., None]
    else:
        q, sc, d = _q6k(w)
        v = (q - 32.0) * (d.double() * sc)[..., None]
    return v.view(w.shape)


_DTYPE = {"f32": torch.float32, "bf16": torch.bfloat16}


class _State:
    """What a program holds before the call; the resident weights go with it."""

    def __init__(self, **kw):
        self.__dict__.update(kw)

    def __del__(self):
        for w in self.__dict__.get("weights", ()):
            w.destroy()


def _rows(g, m, n, dtype="f32"):
    return torch.randn((m, n), generator=g, device="cuda").to(_DTYPE[dtype])


def _layers(case, g):
    """Per layer: seven float weights (q, k, v, o, gate, up, down), two gains, both caches."""
    d, qd, kvd, ffn = 128 * case["heads"], case["heads"] * case["hd"], case["kv_heads"] * case["hd"], case["ffn"]
    shapes = ((qd, d), (kvd, d), (kvd, d), (d, qd), (ffn, d), (ffn, d), (d, ffn))
    for _ in range(case["layers"]):
        ws = [_float_weight(g, o, i) for o, i in shapes]
        gains = [1.0 + 0.1 * _rows(g, 1, d).view(-1) for _ in range(2)]
        caches = [_rows(g, case["cached"] + 1, kvd) for _ in range(2)]
        yield ws, gains, caches


def prepare(case, seed):
    g, op = _gen(seed), case["op"]
    if op in ("linear", "linear_i8", "train"):
        w = _weight(case["fmt"], _float_weight(g, case["out"], case["in"]))
        s = _State(case=case, weights=[w], x=_rows(g, case["m"], case["in"], case.get("x", "f32")))
        if op == "train":
            s.dy = _rows(g, case["m"], case["out"])
        return s
    if op == "encode":
        return _State(case=case, w=_float_weight(g, case["out"], case["in"]))
    if op == "attention":
        kvd = case["kv_heads"] * case["hd"]
        return _State(case=case, q=_rows(g, case["heads"], case["hd"]).view(-1), k=_rows(g, 1, kvd).view(-1),
                      v=_rows(g, 1, kvd).view(-1), kc=_rows(g, case["cached"] + 1, kvd),
                      vc=_rows(g, case["cached"] + 1, kvd))
    stack, caches = [], []
    for ws, gains, cc in _layers(case, g):
        q8 = []
        for w in ws:
            q, d = _q8(w)
            q8.append((_host(q, torch.int8), _host(d)))
        stack.append(DecoderLayer(raster_amd.context(0), q8, *(_host(t) for t in gains), 128 * case["heads"],
                                  case["heads"], case["kv_heads"], case["hd"], case["ffn"]))
        caches.append(cc)
    return _State(case=case, weights=stack, caches=caches, x=_rows(g, 1, 128 * case["heads"]).view(-1))


def run(s):
    case = s.case
    op = case["op"]
    if op == "linear":
        return s.weights[0].matmul(s.x, out_dtype=_DTYPE[case["y"]])
    if op == "linear_i8":
        w = s.weights[0]
        xq, xs, xsum = raster_amd.quantize_act_i8(w.ctx, s.x, case["in"])
        return w.matmul_i8(xq, xs, xsum, out_dtype=_DTYPE[case["y"]])
    if op == "train":
        w = s.weights[0]
        return {"y": w.matmul(s.x), "dx": w.matmul_dx(s.dy)}
    if op == "encode":
        ctx = raster_amd.context(0)
        if case["fmt"] == "q8":
            return raster_amd.q8_quantize(ctx, s.w, case["out"], case["in"])
        if case["fmt"] == "q4k":
            return raster_amd.q4k_of(ctx, s.w, case["out"], case["in"])
        return raster_amd.quantize_weight_q6k(ctx, s.w, case["out"], case["in"])
    if op == "attention":
        out = raster_amd.decode_attention(raster_amd.context(0), s.q, s.k, s.v, s.kc, s.vc, case["cached"],
                                          case["heads"], case["kv_heads"], case["hd"], 1e4, case["hd"] ** -0.5)
        return {"out": out, "kcache": s.kc, "vcache": s.vc}
    h = s.x
    for layer, (kc, vc) in zip(s.weights, s.caches):
        h = layer.step(h, kc, vc, case["cached"])
    return {"h": h, "kcache": [kc for kc, _ in s.caches], "vcache": [vc for _, vc in s.caches]}


# ---- work, tolerance and exact values --------------------------------------------


def _weight_bytes(fmt, out, in_):
    per = {"q8": (32 + 4) / 32, "q4h": (16 + 2) / 32, "q4f": (16 + 4) / 32, "q4k": (128 + 8 + 16) / 256,
           "q6k": (192 + 4 + 16) / 256}[fmt]
    return out * in_ * per


def work(case):
    op = case["op"]
    if op in ("linear", "linear_i8", "train"):
        m, in_, out = case["m"], case["in"], case["out"]
        xb = 2 if case.get("x") == "bf16" else 4
        yb = 2 if case.get("y") == "bf16" else 4
        b, f = m * in_ * xb + m * out * yb + _weight_bytes(case["fmt"], out, in_), 2.0 * m * in_ * out
        if op == "train":  # dy in, dx out; the weight again for the second product
            b, f = 2 * b, 2 * f
        return {"bytes": b, "flops": f}
    if op == "encode":
        n, inp = case["out"] * case["in"], (case["in"] + 255) // 256 * 256 if case["fmt"] == "q4k" else case["in"]
        per = {"q8": 36 / 32, "q4k": 152 / 256, "q6k": (256 + 4 + 16) / 256}[case["fmt"]]
        return {"bytes": 4 * n + case["out"] * inp * per, "flops": 4.0 * n}
    kvd, qd, rows = case["kv_heads"] * case["hd"], case["heads"] * case["hd"], case["cached"] + 1
    b, f = 4 * (2 * rows * kvd + 2 * kvd + 2 * qd), 4.0 * rows * qd
    if op == "decoder":
        d, ffn = 128 * case["heads"], case["ffn"]
        n = d * (2 * qd + 2 * kvd + 3 * ffn)
        b, f = case["layers"] * (b + _weight_bytes("q8", 1, n)) + 8 * d, case["layers"] * (f + 2.0 * n)
    return {"bytes": b, "flops": f}


def tolerance(case):
    """About four times the error against 64 bits measured on an MI355X."""
    op = case["op"]
    if op == "encode":
        return "exact"
    if op == "decoder":  # 6.1e-5: 16-bit block fixed-point activations through two layers
        return {"rel": 2.5e-4}
    if op == "attention":  # 2.4e-7
        return {"rel": 2e-6}
    if op == "linear" and case["x"] == "bf16" or case.get("y") == "bf16":  # 2.3e-3, bf16 operands or result
        return {"rel": 1e-2}
    if op == "train":  # 4.4e-6: dy and w carried as two bf16 terms each
        return {"rel": 2e-5}
    if op == "linear_i8" or case["fmt"] in ("q4k", "q6k"):  # 1.2e-7: exact integer dots, f32 sums
        return {"rel": 2e-6}
    # f32 x: 3.4e-5 with 16-bit block fixed point (m <= 16), 2.5e-6 with two bf16 terms
    return {"rel": 1.3e-4 if case["m"] <= 16 else 1e-5}


def _act_i8(x, n):
    """Activations quantized to int8 blocks of n, as 64-bit values."""
    b = _blocks(x, n)
    d = b.abs().amax(2, keepdim=True) / 127.0
    return (_round(b * _inv(d), -127, 127) * d.float().double()).view(x.shape)


def _rope(t, heads, hd, pos):
    ang = pos * torch.exp(torch.arange(hd // 2, dtype=torch.float64, device="cuda") * (-2.0 / hd) * math.log(1e4))
    a, b = t.view(heads, 2, hd // 2).unbind(1)
    return torch.cat([a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()], 1)


def _attend(case, q, k, v, kc, vc):
    """(out, kc, vc) in 64 bits, the caches with the new row at `cached`."""
    h, kvh, hd, pos = case["heads"], case["kv_heads"], case["hd"], case["cached"]
    kc, vc = kc.double().clone(), vc.double().clone()
    kc[pos], vc[pos] = _rope(k, kvh, hd, pos).view(-1), v
    qr = _rope(q, h, hd, pos)
    out = torch.empty_like(qr)
    for i in range(h):
        j = i // (h // kvh)
        p = torch.softmax(kc[:, j * hd:(j + 1) * hd] @ qr[i] * hd ** -0.5, 0)
        out[i] = p @ vc[:, j * hd:(j + 1) * hd]
    return out.view(-1), kc, vc


def exact(case, seed):
    g, op = _gen(seed), case["op"]
    if op in ("linear", "linear_i8", "train"):
        fmt = case["fmt"]
        w = _dense(fmt, _float_weight(g, case["out"], case["in"]))
        x = _rows(g, case["m"], case["in"], case.get("x", "f32"))
        if op == "linear_i8":
            return _act_i8(x, 32) @ w.T
        if op == "train":
            return {"y": x.double() @ w.T, "dx": _rows(g, case["m"], case["out"]).double() @ w}
        return (_act_i8(x, 256) if fmt in ("q4k", "q6k") else x.double()) @ w.T
    if op == "encode":
        w = _float_weight(g, case["out"], case["in"])
        if case["fmt"] == "q8":
            q, d = _q8(w)
            return q.view(w.shape).to(torch.int8), d.double().squeeze(2)
        if case["fmt"] == "q6k":
            q, sc, d = _q6k(w)
            return q.view(-1).to(torch.uint8), sc.view(-1).to(torch.int8), d.double().view(-1)
        inp = (case["in"] + 255) // 256 * 256
        w = torch.nn.functional.pad(w, (0, inp - case["in"]))
        q, da, db, aq, bq = _q4k(w)
        q = q.to(torch.uint8)
        return {"wq": (q[..., :16] | (q[..., 16:] << 4)).view(-1), "da": da.double().view(-1),
                "db": db.double().view(-1), "aq": aq.to(torch.uint8).view(-1), "bq": bq.to(torch.int8).view(-1),
                "in": inp, "out": case["out"]}
    if op == "attention":
        s = prepare(case, seed)
        out, kc, vc = _attend(case, s.q.double(), s.k.double(), s.v.double(), s.kc, s.vc)
        return {"out": out, "kcache": kc, "vcache": vc}
    layers = list(_layers(case, g))
    h, kcs, vcs = _rows(g, 1, 128 * case["heads"]).view(-1).double(), [], []

    def norm(t, gain):
        return t * torch.rsqrt((t * t).mean() + 1e-5) * gain.double()

    for ws, gains, (kc, vc) in layers:
        wq, wk, wv, wo, wg, wu, wd = (_dense("q8", w) for w in ws)
        t = norm(h, gains[0])
        at, kc, vc = _attend(case, wq @ t, wk @ t, wv @ t, kc, vc)
        h = h + wo @ at
        t = norm(h, gains[1])
        z = wg @ t
        h = h + wd @ (z * torch.sigmoid(z) * (wu @ t))
        kcs.append(kc)
        vcs.append(vc)
    return {"h": h, "kcache": kcs, "vcache": vcs}
