"""The calls that a program built on this library spends its GPU time in.

Each case is one call, or the few calls of one layer, through the entry points
of runtimed_amd.rq, over sizes of this repository's own workloads (a Qwen2-0.5B
shaped layer, a 2048 / 8192 layer with a 262144-row head, 14336 x 4096 streaming
and FP8 weights) and generic ones around them.  The reference computes in f32
and calls a linear with t = 1 rows (decode), 2..16 (speculative verify) or up to
512 (a prefill chunk); bf16 and f16 activations are options of the same calls.

Kinds:
  layer   the quantized linears of one transformer layer (q/k/v with biases and
          gate/up as one call each, then o and down)
  head    the output projection of the last position
  embed   rows of the token embedding, as a prompt looks them up
  dense   a weight decoded to f32 (Weights::get)
  fp8     an e4m3 weight with per-row scales, activations encoded on the fly
  marlin  the INT4 linears of a gated MLP
  kv      a K / V chunk quantized into a cache block and read back
"""
from __future__ import annotations

import math

import torch

from runtimed_amd import rq

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
QTYPES = ("Q4_K", "Q6_K", "Q8_0", "Q5_K", "Q4_0", "Q5_0")
BLOCK = {"Q4_0": (32, 18), "Q5_0": (32, 22), "Q8_0": (32, 34), "Q4_K": (256, 144), "Q5_K": (256, 176),
         "Q6_K": (256, 210)}


def listed():
    return [
        # one decoded token through a 0.5B layer: small launches, latency
        {"name": "decode_layer_896", "kind": "layer", "m": 1, "hidden": 896, "kv": 128, "ffn": 4864,
         "main": "Q4_K", "mixed": "Q4_K", "x": "f32"},
        # one decoded token through a 4096 / 14336 layer in the Q4_K_M mix: weight streaming
        {"name": "decode_layer_4096", "kind": "layer", "m": 1, "hidden": 4096, "kv": 1024, "ffn": 14336,
         "main": "Q4_K", "mixed": "Q6_K", "x": "f32"},
        # the output projection of a decoded token: the largest weight there is
        {"name": "decode_head", "kind": "head", "m": 1, "n": 262144, "k": 2048, "q": "Q6_K", "x": "f32"},
        # eight draft tokens verified in one pass of a 2048 / 8192 layer
        {"name": "verify_layer_2048", "kind": "layer", "m": 8, "hidden": 2048, "kv": 2048, "ffn": 8192,
         "main": "Q4_K", "mixed": "Q6_K", "x": "f32"},
        # a full prefill chunk in the reference's compute type
        {"name": "prefill_layer_f32", "kind": "layer", "m": 512, "hidden": 2048, "kv": 2048, "ffn": 8192,
         "main": "Q4_K", "mixed": "Q6_K", "x": "f32"},
        # the last, ragged chunk of a prompt in bf16, on Q8_0 weights
        {"name": "prefill_ragged_bf16", "kind": "layer", "m": 333, "hidden": 2048, "kv": 512, "ffn": 8192,
         "main": "Q8_0", "mixed": "Q8_0", "x": "bf16"},
        # a prompt's token embeddings
        {"name": "embed_prompt", "kind": "embed", "ids": 512, "n": 151936, "k": 896, "q": "Q8_0"},
        # FP8 decode / verify of a few rows: weight streaming
        {"name": "fp8_verify", "kind": "fp8", "m": 5, "n": 14336, "k": 4096, "x": "f32", "mode": "per_token"},
        # FP8 prefill
        {"name": "fp8_prefill", "kind": "fp8", "m": 2048, "n": 14336, "k": 4096, "x": "bf16", "mode": "per_token"},
        # one decoded token through an INT4 MLP
        {"name": "marlin_decode", "kind": "marlin", "m": 1, "hidden": 4096, "ffn": 14336, "x": "f32"},
        # a prompt chunk through an INT4 MLP
        {"name": "marlin_prefill", "kind": "marlin", "m": 300, "hidden": 2048, "ffn": 8192, "x": "f32"},
        # a prefill's K and V into FP8 cache blocks and back
        {"name": "kv_blocks", "kind": "kv", "heads": 8, "tokens": 4096, "dim": 128, "x": "bf16", "mode": "fp8"},
    ]


# ---- drawn cases ----

# multiply-adds of the listed prefill layer and INT4 prefill: a drawn chunk on wider weights has fewer rows
LAYER_WORK = 512 * 2048 * (4 * 2048 + 3 * 8192)
MLP_WORK = 300 * 3 * 2048 * 8192


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mult(rng, step, lo, hi):
    """A multiple of step, its logarithm uniform in [lo, hi]."""
    return max(lo, _log(rng, lo, hi) // step * step)


def _rows(rng):
    """Rows of a call: a decoded token, a verify step or a prefill chunk."""
    return rng.choice([1, 1, _log(rng, 2, 16), _log(rng, 2, 16), _log(rng, 17, 512), _log(rng, 17, 512)])


def _xtype(rng):
    return rng.choice(["f32", "f32", "bf16", "f16"])


def draw(rng):
    """One more case: rows over 1..512 (FP8 up to 2048), widths over the sizes of 0.5B to 8B models
    (multiples of 128; 1 in 4 FP8 and INT4 widths only of 32), every format and activation type."""
    kind = rng.choice(["layer"] * 5 + ["head", "embed", "dense", "fp8", "fp8", "fp8", "marlin", "marlin", "marlin",
                                       "kv", "kv"])
    if kind == "layer":
        hidden = _mult(rng, 128, 512, 4096)
        main = rng.choice(["Q4_K", "Q4_K", "Q8_0", "Q6_K", "Q5_K", "Q4_0", "Q5_0"])
        kv, ffn = _mult(rng, 64, 128, hidden), _mult(rng, 128, 2 * hidden, 4 * hidden)
        weights = hidden * (2 * hidden + 2 * kv + 3 * ffn)
        return {"kind": kind, "m": min(_rows(rng), LAYER_WORK // weights), "hidden": hidden, "kv": kv,
                "ffn": ffn, "main": main,
                "mixed": "Q6_K" if main in ("Q4_K", "Q5_K") and rng.random() < 0.5 else main, "x": _xtype(rng)}
    if kind == "head":
        return {"kind": kind, "m": rng.choice([1, 1, _log(rng, 2, 16)]), "n": 8 * _log(rng, 4000, 32768),
                "k": _mult(rng, 128, 512, 2048), "q": rng.choice(QTYPES), "x": _xtype(rng)}
    if kind == "embed":
        return {"kind": kind, "ids": _log(rng, 1, 512), "n": 8 * _log(rng, 4000, 32768),
                "k": _mult(rng, 128, 512, 2048), "q": rng.choice(QTYPES)}
    if kind == "dense":
        return {"kind": kind, "n": 8 * _log(rng, 16, 1792), "k": _mult(rng, 128, 512, 4096), "q": rng.choice(QTYPES)}
    if kind == "fp8":
        return {"kind": kind, "m": rng.choice([_rows(rng), _rows(rng), _log(rng, 256, 2048)]),
                "n": _log(rng, 256, 14336), "k": _mult(rng, rng.choice([128, 128, 128, 32]), 512, 4096),
                "x": _xtype(rng), "mode": rng.choice(["per_token", "per_token", "unscaled"])}
    if kind == "marlin":
        step = rng.choice([128, 128, 128, 32])
        hidden = _mult(rng, step, 512, 4096)
        ffn = _mult(rng, step, 2 * hidden, 4 * hidden)
        return {"kind": kind, "m": min(_rows(rng), MLP_WORK // (3 * hidden * ffn)), "hidden": hidden, "ffn": ffn,
                "x": _xtype(rng)}
    return {"kind": kind, "heads": rng.choice([2, 4, 8, 16]), "tokens": _log(rng, 16, 4096),
            "dim": rng.choice([64, 80, 128]), "x": rng.choice(["f32", "bf16", "f16"]),
            "mode": rng.choice(["fp8", "fp8", "int8"])}


# ---- inputs ----

DEVICE = "cuda"


class Draws:
    """Seeded tensors on the GPU."""

    def __init__(self, seed: int):
        self.g = torch.Generator(device=DEVICE)
        self.g.manual_seed(int(seed))

    def normal(self, *shape):
        return torch.randn(shape, generator=self.g, device=DEVICE)

    def ints(self, lo, hi, *shape):
        return torch.randint(lo, hi, shape, generator=self.g, device=DEVICE, dtype=torch.int32)

    def uniform(self, lo, hi, *shape):
        return torch.rand(shape, generator=self.g, device=DEVICE) * (hi - lo) + lo

    def codes(self, mid, dev, lo, hi, *shape):
        """Codes of a normal weight: round(N(mid, dev)) within [lo, hi]."""
        return (self.normal(*shape).mul_(dev).add_(mid)).round_().clamp_(lo, hi).to(torch.int16)


def _f16_bytes(v):
    return v.to(torch.float16).view(torch.uint8).reshape(v.shape[0], -1)


def _u8(v):
    return v.to(torch.uint8)


def _k_scales(sc, mn):
    """The 12 scale bytes of a Q4_K / Q5_K block from eight 6-bit scales and mins."""
    out = torch.empty((sc.shape[0], 12), dtype=torch.int32, device=sc.device)
    out[:, 0:4] = sc[:, 0:4] | ((sc[:, 4:8] >> 4) << 6)
    out[:, 4:8] = mn[:, 0:4] | ((mn[:, 4:8] >> 4) << 6)
    out[:, 8:12] = (sc[:, 4:8] & 15) | ((mn[:, 4:8] & 15) << 4)
    return _u8(out)


def make_blocks(d: Draws, q: str, n: int, k: int):
    """(GGUF blocks as a uint8 tensor, function that gives the f64 weight [n, k]) of a normal weight."""
    nb = n * k // BLOCK[q][0]
    step = 0.02 * 3.0  # the weights' spread
    if q in ("Q4_K", "Q5_K"):
        top = 15 if q == "Q4_K" else 31
        sc = d.ints(30, 64, nb, 8)
        mn = (sc + d.ints(-2, 3, nb, 8)).clamp_(0, 63)
        dd = (d.uniform(0.8, 1.2, nb, 1) * (step / (top / 2) / 48)).to(torch.float16)
        dm = (dd.float() * (top / 2)).to(torch.float16)
        c = d.codes(top / 2, top / 6, 0, top, nb, 8, 32)  # sub-block j: elements 32 j .. 32 j + 31
        lo = _u8((c[:, 0::2] & 15) | ((c[:, 1::2] & 15) << 4)).reshape(nb, 128)
        parts = [_f16_bytes(dd), _f16_bytes(dm), _k_scales(sc, mn)]
        if q == "Q5_K":
            bits = torch.arange(8, device=c.device, dtype=torch.int16).view(1, 8, 1)
            parts.append(_u8(((c >> 4) << bits).sum(1)))
        raw = torch.cat(parts + [lo], 1)

        def value():
            return ((dd.double() * sc.double()).unsqueeze(2) * c.double() - (dm.double() * mn.double()).unsqueeze(2)
                    ).reshape(n, k)
    elif q == "Q6_K":
        sc = d.ints(40, 128, nb, 16) * (2 * d.ints(0, 2, nb, 16) - 1)
        dd = (d.uniform(0.8, 1.2, nb, 1) * (step / 32 / 84)).to(torch.float16)
        c = d.codes(32, 10.7, 0, 63, nb, 2, 4, 32)  # element 128 h + 32 t + l
        ql = _u8(torch.cat([(c[:, :, 0] & 15) | ((c[:, :, 2] & 15) << 4), (c[:, :, 1] & 15) | ((c[:, :, 3] & 15) << 4)],
                           2)).reshape(nb, 128)
        qh = _u8((c[:, :, 0] >> 4) | ((c[:, :, 1] >> 4) << 2) | ((c[:, :, 2] >> 4) << 4) | ((c[:, :, 3] >> 4) << 6)
                 ).reshape(nb, 64)
        raw = torch.cat([ql, qh, sc.to(torch.int8).view(torch.uint8), _f16_bytes(dd)], 1)

        def value():
            s = (dd.double() * sc.double()).unsqueeze(2)  # 16 runs of 16 elements
            return (s * (c.reshape(nb, 16, 16).double() - 32.0)).reshape(n, k)
    else:
        half = {"Q8_0": 0, "Q4_0": 8, "Q5_0": 16}[q]
        span = half or 127
        dd = (d.uniform(0.8, 1.2, nb, 1) * (step / span)).to(torch.float16)
        c = d.codes(half, span / 3, half - span, half + span - (1 if half else 0), nb, 32)
        if q == "Q8_0":
            raw = torch.cat([_f16_bytes(dd), c.to(torch.int8).view(torch.uint8)], 1)
        else:
            parts = [_f16_bytes(dd)]
            if q == "Q5_0":
                bits = torch.arange(8, device=c.device, dtype=torch.int16).view(1, 1, 8)
                parts.append(_u8(((c >> 4).reshape(nb, 4, 8) << bits).sum(2)))
            raw = torch.cat(parts + [_u8((c[:, :16] & 15) | ((c[:, 16:] & 15) << 4))], 1)

        def value():
            return (dd.double() * (c.double() - half)).reshape(n, k)
    return raw.reshape(-1), value


def _linears(case):
    """(name, rows, width, format, has a bias) of a layer's weights."""
    h, kv, f = case["hidden"], case["kv"], case["ffn"]
    a, b = case["main"], case["mixed"]
    return [("q", h, h, a, True), ("k", kv, h, a, True), ("v", kv, h, b, True), ("o", h, h, a, False),
            ("gate", f, h, a, False), ("up", f, h, a, False), ("down", h, f, b, False)]


# (weights of one call, input of that call) in the order of a layer's forward pass
LAYER_CALLS = ((("q", "k", "v"), "attn_in"), (("o",), "attn_out"), (("gate", "up"), "mlp_in"), (("down",), "mlp_mid"))
MLP_CALLS = ((("gate",), "mlp_in"), (("up",), "mlp_in"), (("down",), "mlp_mid"))


def _inputs(case, seed):
    """Everything that prepare and exact share: raw weights, their f64 values and the activations."""
    d, kind = Draws(seed), case["kind"]
    s = {}
    if kind == "layer":
        dt, m = DTYPES[case["x"]], case["m"]
        s["w"] = {nm: make_blocks(d, q, n, k) + (q, n, k) for nm, n, k, q, _ in _linears(case)}
        s["b"] = {nm: d.normal(n).mul_(0.1) for nm, n, _, _, bias in _linears(case) if bias}
        s["x"] = {nm: d.normal(1, m, case["ffn"] if nm == "mlp_mid" else case["hidden"]).to(dt)
                  for _, nm in LAYER_CALLS}
    elif kind in ("head", "embed", "dense"):
        s["w"] = make_blocks(d, case["q"], case["n"], case["k"]) + (case["q"], case["n"], case["k"])
        if kind == "head":
            s["x"] = d.normal(1, case["m"], case["k"]).to(DTYPES[case["x"]])
        elif kind == "embed":
            s["ids"] = d.ints(0, case["n"], case["ids"]).cpu().numpy().astype("uint32")
    elif kind == "fp8":
        w = d.normal(case["n"], case["k"]).clamp_(-448.0, 448.0).to(torch.float8_e4m3fn)
        s["w"], s["ws"] = w.view(torch.uint8), d.uniform(0.5, 2.0, case["n"]) / 448.0
        s["x"] = d.normal(1, case["m"], case["k"]).to(DTYPES[case["x"]])
    elif kind == "marlin":
        h, f = case["hidden"], case["ffn"]
        s["w"] = {}
        for nm, n, k in (("gate", f, h), ("up", f, h), ("down", h, f)):
            c = d.codes(8, 2.5, 0, 15, n, k)
            shift = 4 * torch.arange(8, device=DEVICE, dtype=torch.int64)
            words = torch.empty((n, k // 32, 4), dtype=torch.int32, device=DEVICE)
            for r in range(0, n, 4096):  # bounded scratch
                w64 = (c[r:r + 4096].reshape(-1, k // 32, 4, 8).long() << shift).sum(3)
                words[r:r + 4096] = torch.where(w64 >= 1 << 31, w64 - (1 << 32), w64).to(torch.int32)
            s["w"][nm] = (words.permute(1, 0, 2).contiguous(), d.uniform(0.5, 1.5, n) * 0.008, c, n, k)
        s["x"] = {nm: d.normal(1, case["m"], f if nm == "mlp_mid" else h).to(DTYPES[case["x"]])
                  for nm in ("mlp_in", "mlp_mid")}
    else:
        shape = (1, case["heads"], case["tokens"], case["dim"])
        s["k"], s["v"] = (d.normal(*shape).to(DTYPES[case["x"]]) for _ in range(2))
    return s


def _qweight(raw, value, q, n, k):
    return rq.QWeight(rq.QTYPES[q], raw.cpu().numpy(), n, k)


def prepare(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    s["case"] = case
    if kind == "layer":
        s["w"] = {nm: _qweight(*w) for nm, w in s["w"].items()}
    elif kind in ("head", "embed", "dense"):
        s["w"] = _qweight(*s["w"])
    elif kind == "marlin":
        s["w"] = {nm: rq.MarlinWeight(p, sc, k, n) for nm, (p, sc, _, n, k) in s["w"].items()}
    return s


# ---- one pass ----

def run(state):
    case, w = state["case"], state.get("w")
    kind = case["kind"]
    if kind == "layer":
        x, b = state["x"], state["b"]
        out = {}
        for names, src in LAYER_CALLS:
            if len(names) > 1:
                biases = [b[nm] for nm in names] if names[0] in b else None
                out.update(zip(names, rq.linear_multi([w[nm] for nm in names], x[src], biases)))
            else:
                out[names[0]] = w[names[0]].forward(x[src])
        return out
    if kind == "head":
        return w.forward(state["x"], out_dtype=torch.float32)
    if kind == "embed":
        return w.embedding(state["ids"])
    if kind == "dense":
        return w.dequantize()
    if kind == "fp8":
        mode = rq.FP8_PER_TOKEN if case["mode"] == "per_token" else rq.FP8_UNSCALED
        return rq.fp8_gemm(state["x"], w, state["ws"], mode=mode, out_dtype=state["x"].dtype)
    if kind == "marlin":
        return {nm: rq.marlin_gemv(state["x"][src], w[nm]) for (nm,), src in MLP_CALLS}
    # one block past the attention sink, written and read back for attention
    prec = rq.KV_FP8 if case["mode"] == "fp8" else rq.KV_INT8
    kq, vq, ks, vs, mode = rq.quantize_block_kv(rq.SINK_TOKENS_COUNT, state["k"], state["v"], prec)
    dt = state["k"].dtype
    return {"kq": kq.view(torch.uint8), "vq": vq.view(torch.uint8), "ks": ks, "vs": vs,
            "k": rq.dequantize_block(kq, ks, mode, dt), "v": rq.dequantize_block(vq, vs, mode, dt)}


# ---- what a pass cannot do without ----

def _qbytes(q, n, k):
    return n * k // BLOCK[q][0] * BLOCK[q][1]


def work(case):
    kind = case["kind"]
    xb = DTYPES[case["x"]].itemsize if "x" in case else 4
    if kind == "layer":
        m, nbytes, flops = case["m"], 0, 0
        for nm, n, k, q, bias in _linears(case):
            nbytes += _qbytes(q, n, k) + (4 * n if bias else 0) + m * n * xb
            flops += 2 * m * n * k
        nbytes += m * xb * (3 * case["hidden"] + case["ffn"])  # each input once
        return {"bytes": nbytes, "flops": flops}
    if kind == "head":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": _qbytes(case["q"], n, k) + m * k * xb + m * n * 4, "flops": 2 * m * n * k}
    if kind == "embed":
        return {"bytes": _qbytes(case["q"], 1, case["k"] * case["ids"]) + case["ids"] * (4 * case["k"] + 4),
                "flops": case["ids"] * case["k"]}
    if kind == "dense":
        n, k = case["n"], case["k"]
        return {"bytes": _qbytes(case["q"], n, k) + 4 * n * k, "flops": n * k}
    if kind == "fp8":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": n * k + 4 * n + m * (n + k) * xb, "flops": 2 * m * n * k}
    if kind == "marlin":
        m, h, f = case["m"], case["hidden"], case["ffn"]
        return {"bytes": 3 * h * f // 2 + 4 * (2 * f + h) + m * (2 * h + 3 * f) * xb, "flops": 6 * m * h * f}
    e = 2 * case["heads"] * case["tokens"] * case["dim"]
    return {"bytes": e * (2 * xb + 1) + 8 * case["heads"], "flops": 4 * e}


# ---- tolerances ----

def tolerance(case):
    """Decoded rows, codes and cache blocks are fixed by the formats, bit for bit.  Sums (measured against 64 bits,
    times four): f32 activations run on exact f32 products or on two 16-bit limbs, 6e-6; the fp8 matrix cores' own
    sums, 1.4e-5; bf16 activations with weights and results rounded to bf16, 2.9e-3, f16 results 3e-4."""
    kind = case["kind"]
    if kind in ("embed", "dense", "kv"):
        return "exact"
    if case["x"] == "f32":
        return {"rel": 6e-5 if kind == "fp8" else 2.5e-5}
    return {"rel": 1.2e-2 if case["x"] == "bf16" else 1.2e-3}


# ---- the same in 64 bits ----

def _mm(x, w):
    return x.double() @ w.t()


def _e4m3_nearest(v):
    """The nearest e4m3 value, ties to the lower magnitude, saturating at 448, in f64."""
    a = v.double().abs().clamp(max=448.0)
    e = torch.floor(torch.log2(a.clamp(min=2.0 ** -6))).clamp(-6, 8)
    ulp = torch.exp2(e - 3)
    r = torch.ceil(a / ulp - 0.5) * ulp
    return torch.copysign(r.clamp(max=448.0), v.double())


def exact(case, seed):
    kind = case["kind"]
    s = _inputs(case, seed)
    if kind == "layer":
        out = {}
        for names, src in LAYER_CALLS:
            for nm in names:
                y = _mm(s["x"][src], s["w"][nm][1]())
                out[nm] = y + s["b"][nm].double() if nm in s["b"] else y
        return out
    if kind == "head":
        value, n, k = s["w"][1], case["n"], case["k"]
        return _mm(s["x"], value())
    if kind == "embed":
        ids = torch.from_numpy(s["ids"].astype("int64")).to(DEVICE)
        return s["w"][1]()[ids]
    if kind == "dense":
        return s["w"][1]()
    if kind == "fp8":
        x = s["x"].float()
        w = s["w"].view(torch.float8_e4m3fn).double() * s["ws"].double().unsqueeze(1)
        if case["mode"] == "unscaled":
            return _mm(_e4m3_nearest(x), w)
        amax = x.abs().amax(-1, keepdim=True)
        codes = (x * (torch.full_like(amax, 448.0) / amax)).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
        return _mm(codes.double() * (amax.double() / 448.0), w)
    if kind == "marlin":
        return {nm: _mm(s["x"][src], (s["w"][nm][2].double() - 8.0) * s["w"][nm][1].double().unsqueeze(1))
                for (nm,), src in MLP_CALLS}
    top = 448.0 if case["mode"] == "fp8" else 127.0
    out = dict.fromkeys(("kq", "vq", "ks", "vs", "k", "v"))
    for nm in ("k", "v"):
        out[nm + "s"] = (s[nm].double().abs().amax((0, 2, 3), keepdim=True) / top).clamp(min=1e-8)
    return out
