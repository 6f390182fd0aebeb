"""Performance cases of the quantized product library, through its Python binding.

What a program that serves a GGUF model asks of the library, over the whole
range of each call: single projections at decode, the same projections for a
few sequences at once and for the positions of a prefill step, the gguf_moe
block at one position and over a prefill batch, recipe's int(8) sum, and a
whole decode step replayed from a captured graph.

A case is a dict; `kind` says which call it is:
  product  y = W x for m activation rows of fp16 or fp32 (Weight.matvec)
  moe      one gguf_moe block over m positions (Moe.run / Moe.run_batch)
  int8     recipe's int(8) sum over m fp32 rows (matvec_int8)
  decode   one token of a llama-style decoder (DecodeModel, captured graph)

Weights and activations follow the synthetic workload definitions of
rqmv.synth (block codes uniform over their range, half-normal fp16 block
scales, activations N(0,1), router N(0, 0.02)), with the block scales brought
to where a weight's standard deviation is about 0.05, so that the activations
inside a MoE block and through a decoder's layers keep the magnitudes that a
trained model's have. Everything is drawn on the device from the seed.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "recipe-dev_amd"))

import rqmv  # noqa: E402
from rqmv import decode as rqdecode  # noqa: E402

# (values, bytes) of one GGUF block
BLOCK = {"q4_0": (32, 18), "q8_0": (32, 34), "q4_k": (256, 144), "q6_k": (256, 210)}
FORMATS = sorted(BLOCK)
# standard deviation of the normal whose magnitude is a block's fp16 scale
SCALE = {"q4_0": 0.01, "q8_0": 6e-4, "q4_k": 1.6e-4, "q6_k": 1.5e-4}

# The largest product of the range: 512 positions through an FFN projection.
MOST_MACS = 512 * 14336 * 4096
MOST_WEIGHTS = 25600 * 5120
# The largest block of a MoE draw (weights of the bank) and of a decoder draw.
MOST_BANK = 256 * 3 * 512 * 2048


# ------------------------------------------------------------------ cases ----

def product(name, fmt, rows, cols, m, x):
    return {"name": name, "kind": "product", "fmt": fmt, "rows": rows, "cols": cols, "m": m, "x": x}


def listed():
    return [
        # the smallest projection of a grouped-query layer (8 kv heads of 128) for one token
        product("kv_proj_decode", "q4_k", 1024, 4096, 1, "f32"),
        # the FFN gate/up projection for one token: the headline configuration
        product("ffn_up_decode", "q4_k", 14336, 4096, 1, "f16"),
        # the FFN down projection for one token, long rows, fp32 activations as the decode step has them
        product("ffn_down_decode", "q4_0", 4096, 14336, 1, "f32"),
        # verification of a few speculated tokens: an odd row count, fp32 activations
        product("verify_5_rows", "q4_k", 4096, 4096, 5, "f32"),
        # eight sequences decoded together, the largest single weight
        product("q6_batch_8", "q6_k", 25600, 5120, 8, "f16"),
        # thirty-two sequences decoded together
        product("q8_batch_32", "q8_0", 5120, 5120, 32, "f16"),
        # a prefill step of 512 positions through an FFN projection
        product("prefill_512", "q4_k", 14336, 4096, 512, "f16"),
        # a short prompt: ragged positions, long rows, fp32 activations
        product("prefill_77", "q6_k", 4096, 14336, 77, "f32"),
        # a gguf_moe block for one token: 256 experts of 512, top 8, a gated shared expert
        {"name": "moe_decode", "kind": "moe", "fmt": "q4_k", "d": 2048, "hidden": 512, "experts": 256, "top": 8,
         "shared": True, "m": 1, "x": "f16"},
        # the same block over the positions of a prefill step
        {"name": "moe_prefill", "kind": "moe", "fmt": "q4_k", "d": 2048, "hidden": 512, "experts": 256, "top": 8,
         "shared": True, "m": 512, "x": "f16"},
        # recipe's default precision profile (int8 sum, step 32) for four sequences
        {"name": "int8_batch_4", "kind": "int8", "fmt": "q4_k", "rows": 14336, "cols": 4096, "m": 4, "step": 32},
        # four layers and the head of the 32-layer decoder at context 4096
        {"name": "decode_step", "kind": "decode", "layers": 4, "d": 4096, "q_heads": 32, "kv_heads": 8,
         "head_dim": 128, "ffn": 14336, "vocab": 32768, "ctx": 4096, "fmt": "q4_k", "head": "q8_0"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("product", "product", "product", "moe", "int8", "decode"))
    if kind in ("product", "int8"):
        fmt = rng.choice(FORMATS if kind == "product" else ("q4_k", "q8_0"))
        unit = 32 if fmt in ("q4_0", "q8_0") else 256
        while True:
            rows = _log(rng, 256, 25600)
            cols = max(1, _log(rng, 1024, 14336) // unit) * unit
            m = _log(rng, 1, 512 if kind == "product" else 16)
            if rows * cols <= MOST_WEIGHTS and rows * cols * m <= MOST_MACS:
                break
        if kind == "int8":
            step = 32 if cols % 256 else rng.choice((32, 256))
            return {"kind": kind, "fmt": fmt, "rows": rows, "cols": cols, "m": m, "step": step}
        return {"kind": kind, "fmt": fmt, "rows": rows, "cols": cols, "m": m, "x": rng.choice(("f16", "f32"))}
    if kind == "moe":
        while True:
            case = {"kind": kind, "fmt": rng.choice(("q4_k", "q4_k", "q6_k", "q8_0", "q4_0")),
                    "d": rng.choice((1024, 1536, 2048)), "hidden": rng.choice((256, 512, 768)),
                    "experts": rng.choice((32, 60, 64, 128, 256)), "top": rng.choice((2, 4, 6, 8)),
                    "shared": rng.random() < 0.5, "m": _log(rng, 1, 512), "x": rng.choice(("f16", "f32"))}
            if 3 * case["experts"] * case["hidden"] * case["d"] <= MOST_BANK:
                return case
    kv = rng.choice((2, 4, 8))
    group = rng.choice((2, 4, 8))
    hd = 128 if kv * group * 128 <= 4096 else 64
    return {"kind": "decode", "layers": rng.randint(1, 4), "d": kv * group * hd, "q_heads": kv * group,
            "kv_heads": kv, "head_dim": hd, "ffn": 256 * rng.randint(8, 56), "vocab": _log(rng, 4000, 32768),
            "ctx": _log(rng, 16, 8192), "fmt": rng.choice(("q4_k", "q4_0", "q8_0")),
            "head": rng.choice(("q6_k", "q8_0"))}


# ----------------------------------------------------------------- inputs ----

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _bytes(n, cols, g):
    return torch.randint(0, 256, (n, cols), dtype=torch.uint8, device="cuda", generator=g)


def _scale(n, std, g):
    return (torch.randn(n, 1, device="cuda", generator=g).abs() * std).half().view(torch.uint8)


def blocks(fmt, rows, cols, g):
    """GGUF blocks of rows x cols weights, [blocks, block bytes], on the device."""
    values, size = BLOCK[fmt]
    n = rows * (cols // values)
    b = _bytes(n, size, g)
    if fmt == "q6_k":
        b[:, 192:208] = torch.randint(-32, 32, (n, 16), dtype=torch.int8, device="cuda", generator=g).view(torch.uint8)
        b[:, 208:] = _scale(n, SCALE[fmt], g)
        return b
    if fmt == "q8_0":
        b[:, 2:] = torch.randint(-127, 128, (n, 32), dtype=torch.int8, device="cuda", generator=g).view(torch.uint8)
    b[:, :2] = _scale(n, SCALE[fmt], g)
    if fmt == "q4_k":
        b[:, 2:4] = _scale(n, 8 * SCALE[fmt], g)  # minimums about as large as half a code's range
    return b


def _x(m, cols, kind, g):
    x = torch.randn(m, cols, device="cuda", generator=g)
    return x.half() if kind == "f16" else x


def _f16_weight(rows, cols, g):
    return (torch.randn(rows, cols, device="cuda", generator=g) * 0.02).half()


def _norm(n, g):
    return 1.0 + 0.1 * torch.randn(n, device="cuda", generator=g)


def _host(t):
    return t.cpu().numpy()


def _buf(t):
    """A tensor's memory as the binding takes device memory."""
    return rqmv.BufferView(t, t.data_ptr(), t.numel() * t.element_size())


class _Foreign:
    """Device memory of the binding as torch takes foreign memory."""

    def __init__(self, buf, shape, typestr):
        self.keep = buf
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (buf.ptr, False), "version": 2}


def _tensor(buf, shape, typestr):
    return torch.as_tensor(_Foreign(buf, shape, typestr), device="cuda")


_ready = []


def _stream():
    """The program's own stream (graphs are not captured on the default one)."""
    if not _ready:
        rqmv.init(0)
        _ready.append(rqmv.Stream())
    return _ready[0]


# ---------------------------------------------------------------- prepare ----

def _moe_inputs(case, g):
    d, h, e = case["d"], case["hidden"], case["experts"]
    t = {"router": _f16_weight(e, d, g), "gate": blocks(case["fmt"], e * h, d, g),
         "up": blocks(case["fmt"], e * h, d, g), "down": blocks(case["fmt"], e * d, h, g)}
    if case["shared"]:
        t.update(sg=_f16_weight(1, d, g), gs=blocks(case["fmt"], h, d, g), us=blocks(case["fmt"], h, d, g),
                 ds=blocks(case["fmt"], d, h, g))
    t["x"] = _x(case["m"], d, case["x"], g)
    return t


def _decode_inputs(case, g):
    d, ffn, f = case["d"], case["ffn"], case["fmt"]
    kv, hd, ctx = case["kv_heads"], case["head_dim"], case["ctx"]
    layers = []
    for _ in range(case["layers"]):
        layers.append({"qkv": blocks(f, (case["q_heads"] + 2 * kv) * hd, d, g), "o": blocks(f, d, d, g),
                       "gate": blocks(f, ffn, d, g), "up": blocks(f, ffn, d, g), "down": blocks(f, d, ffn, g),
                       "attn_norm": _norm(d, g), "ffn_norm": _norm(d, g),
                       "k": torch.randn(kv, ctx, hd, device="cuda", generator=g).half(),
                       "v": torch.randn(kv, ctx, hd, device="cuda", generator=g).half()})
    return {"layers": layers, "out_norm": _norm(d, g), "head": blocks(case["head"], case["vocab"], d, g),
            "embed": torch.randn(case["vocab"], d, device="cuda", generator=g)}


def prepare(case, seed):
    stream, g, kind = _stream(), _gen(seed), case["kind"]
    if kind in ("product", "int8"):
        rows, cols, m = case["rows"], case["cols"], case["m"]
        make = rqmv.Weight if kind == "product" else rqmv.int8_weight
        w = make(case["fmt"], rows, cols, _host(blocks(case["fmt"], rows, cols, g)))
        x = _x(m, cols, case.get("x", "f32"), g)
        y = torch.empty(m, rows, device="cuda")
        return {"kind": kind, "w": w, "x": _buf(x), "y": y, "out": _buf(y), "m": m, "rows": rows, "cols": cols,
                "dtype": rqmv.DTYPE_F16 if case.get("x") == "f16" else rqmv.DTYPE_F32, "step": case.get("step")}
    if kind == "moe":
        d, h, e, m, fmt = case["d"], case["hidden"], case["experts"], case["m"], case["fmt"]
        t = _moe_inputs(case, g)
        shared = {}
        if case["shared"]:
            shared = {"shared_gate_inp": rqmv.Weight("f16", 1, d, _host(t["sg"])),
                      "gate_sh": rqmv.Weight(fmt, h, d, _host(t["gs"])),
                      "up_sh": rqmv.Weight(fmt, h, d, _host(t["us"])),
                      "down_sh": rqmv.Weight(fmt, d, h, _host(t["ds"]))}
        moe = rqmv.Moe(rqmv.Weight("f16", e, d, _host(t["router"])), rqmv.Weight(fmt, h, d, _host(t["gate"]), experts=e),
                       rqmv.Weight(fmt, h, d, _host(t["up"]), experts=e),
                       rqmv.Weight(fmt, d, h, _host(t["down"]), experts=e), case["top"], **shared)
        y = torch.empty(m, d, device="cuda")
        route = torch.empty(m, e, device="cuda")
        return {"kind": kind, "moe": moe, "x": _buf(t["x"]), "y": y, "route": route, "out": _buf(y),
                "weights": _buf(route), "ws": moe.batch_workspace(m), "m": m, "d": d,
                "dtype": rqmv.DTYPE_F16 if case["x"] == "f16" else rqmv.DTYPE_F32}
    t = _decode_inputs(case, g)
    shape = rqdecode.DecoderShape(layers=case["layers"], d=case["d"], q_heads=case["q_heads"],
                                  kv_heads=case["kv_heads"], head_dim=case["head_dim"], ffn=case["ffn"],
                                  vocab=case["vocab"], proj_fmt=case["fmt"], head_fmt=case["head"])
    model = rqdecode.DecodeModel(shape, case["ctx"] + 64, _host(t["embed"]), _host(t["out_norm"]), _host(t["head"]))
    for i, layer in enumerate(t["layers"]):
        a = {k: _host(layer[k]) for k in ("attn_norm", "qkv", "o", "ffn_norm", "gate", "up", "down")}
        model.set_layer(i, rqdecode.LayerTensors(**a))
        model.set_cache(i, _host(layer["k"]).view(np.uint16), _host(layer["v"]).view(np.uint16))
    token = int(seed) % case["vocab"]
    model.set_position(token, case["ctx"])
    # the prompt's end, to which each pass takes the sequence back
    at = [rqmv.DeviceBuffer.from_array(np.array([v], np.int32)) for v in (token, case["ctx"])]
    cache = (case["kv_heads"], model.max_ctx, case["head_dim"])
    out = {"logits": _tensor(model.logits, (case["vocab"],), "<f4"), "token": _tensor(model.token, (1,), "<i4")}
    for i in range(case["layers"]):  # the appended keys and values
        out["k%d" % i] = _tensor(model.k_cache[i], cache, "<f2")[:, case["ctx"]]
        out["v%d" % i] = _tensor(model.v_cache[i], cache, "<f2")[:, case["ctx"]]
    return {"kind": kind, "model": model, "graph": model.capture(stream), "stream": stream, "at": at, "out": out}


# -------------------------------------------------------------------- run ----

def run(s):
    kind = s["kind"]
    if kind == "product":
        s["w"].matvec(s["x"], s["dtype"], s["m"], s["cols"], s["out"], s["rows"])
        return s["y"]
    if kind == "int8":
        rqmv.matvec_int8(s["w"], s["x"], s["m"], s["cols"], s["out"], s["rows"], s["step"])
        return s["y"]
    if kind == "moe":
        if s["m"] == 1:
            s["moe"].run(s["x"], s["dtype"], s["out"], s["weights"])
        else:
            s["moe"].run_batch(s["x"], s["dtype"], s["m"], s["d"], s["out"], s["d"], s["weights"], s["ws"])
        return {"y": s["y"], "route": s["route"]}
    model, stream = s["model"], s["stream"]
    model.token.copy_from(s["at"][0], 4, stream)
    model.pos.copy_from(s["at"][1], 4, stream)
    s["graph"].launch(stream)
    return s["out"]


# ------------------------------------------------------------------- work ----

def _gguf(fmt, rows, cols):
    values, size = BLOCK[fmt]
    return rows * (cols // values) * size


def work(case):
    kind = case["kind"]
    if kind in ("product", "int8"):
        m, rows, cols = case["m"], case["rows"], case["cols"]
        xsize = 2 if case.get("x") == "f16" else 4
        return {"bytes": _gguf(case["fmt"], rows, cols) + m * cols * xsize + m * rows * 4, "flops": 2.0 * m * rows * cols}
    if kind == "moe":
        d, h, e, m, top, fmt = (case[k] for k in ("d", "hidden", "experts", "m", "top", "fmt"))
        hit = e * (1.0 - (1.0 - top / e) ** m)  # experts that some position selects, on average
        shared = 1 if case["shared"] else 0
        xsize = 2 if case["x"] == "f16" else 4
        return {"bytes": e * d * 2 + shared * d * 2 + (hit + shared) * (2 * _gguf(fmt, h, d) + _gguf(fmt, d, h)) +
                m * (d * xsize + d * 4 + e * 4),
                "flops": float(m) * (2 * e * d + shared * 2 * d + (top + shared) * 6 * h * d)}
    d, ffn, n = case["d"], case["ffn"], case["layers"]
    kv, hd, ctx, vocab = case["kv_heads"], case["head_dim"], case["ctx"], case["vocab"]
    qkv = (case["q_heads"] + 2 * kv) * hd
    proj = _gguf(case["fmt"], qkv, d) + _gguf(case["fmt"], d, d) + 2 * _gguf(case["fmt"], ffn, d) + _gguf(case["fmt"], d, ffn)
    cache = 2 * kv * hd * 2 * (ctx + 1)
    macs = n * ((qkv + d + 3 * ffn) * d + 2 * case["q_heads"] * hd * (ctx + 1)) + vocab * d
    return {"bytes": n * (proj + cache + 8 * d) + _gguf(case["head"], vocab, d) + 4 * d + 4 * d + 4 * vocab,
            "flops": 2.0 * macs}


def tolerance(case):
    kind = case["kind"]
    if kind == "int8":
        return "exact"  # the bits of recipe's int(8) sum
    if kind == "moe":
        return {"rel": 2.5e-4}  # 16-bit activation codes, twice in a row
    if kind == "decode":
        # keys and values are rounded to fp16, where a last-bit difference may flip
        return {"rel": 1e-3}
    # up to four rows the activations are 16-bit integers per block; above, products of exact
    # weight codes and the activations are summed in 32 bits
    return {"rel": 1e-4} if case["m"] <= 4 else {"rel": 1e-5}


# ------------------------------------------------------------------ exact ----

def _f16(b):
    return b.contiguous().view(torch.float16).double()


def dequantize(fmt, b, rows, cols):
    """rows x cols weights in 64 bits from GGUF blocks."""
    n = b.shape[0]
    if fmt == "q8_0":
        w = _f16(b[:, :2]) * b[:, 2:].contiguous().view(torch.int8).double()
    elif fmt == "q4_0":
        w = _f16(b[:, :2]) * (torch.cat((b[:, 2:] & 15, b[:, 2:] >> 4), 1).double() - 8.0)
    elif fmt == "q4_k":
        s = b[:, 4:16]
        sc = torch.cat((s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)), 1).double()
        mn = torch.cat((s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)), 1).double()
        q = b[:, 16:].reshape(n, 4, 1, 32)
        q = torch.cat((q & 15, q >> 4), 2).reshape(n, 8, 32).double()
        w = (_f16(b[:, :2]) * sc).unsqueeze(2) * q - (_f16(b[:, 2:4]) * mn).unsqueeze(2)
    else:
        lo, hi = b[:, :128].reshape(n, 2, 2, 32), b[:, 128:192].reshape(n, 2, 1, 32)
        q = torch.cat(((lo & 15), (lo >> 4)), 2) | torch.cat([((hi >> (2 * i)) & 3) << 4 for i in range(4)], 2)
        scale = _f16(b[:, 208:]) * b[:, 192:208].contiguous().view(torch.int8).double()
        w = scale.unsqueeze(2) * (q.reshape(n, 16, 16).double() - 32.0)
    return w.reshape(rows, cols)


def _records(x, step):
    """The values that recipe's Q8 activation records hold, in 64 bits: codes
    rounded in 32 bits from the inverse step -127 / extreme."""
    v = x.cpu().numpy().reshape(x.shape[0], -1, step)
    at = np.abs(v).argmax(2)
    extreme = np.take_along_axis(v, at[:, :, None], 2)
    inverse = np.float32(-127.0) / extreme
    codes = np.clip(np.rint(v * inverse), -127, 127).astype(np.float64)
    steps = (np.float32(1.0) / inverse).astype(np.float64)
    return torch.from_numpy((codes * steps).reshape(x.shape)).to(x.device)


def _silu(v):
    return v * (0.5 * (torch.tanh(v / 2) + 1.0))


def _exact_moe(case, g):
    t, fmt = _moe_inputs(case, g), case["fmt"]
    d, h, e, m = case["d"], case["hidden"], case["experts"], case["m"]
    x = t["x"].double()
    logits = x @ t["router"].double().t()
    best = torch.sort(logits, dim=1, descending=True, stable=True).indices[:, :case["top"]]
    route = torch.zeros(m, e, dtype=torch.float64, device="cuda")
    route.scatter_(1, best, torch.softmax(torch.gather(logits, 1, best), 1))
    y = torch.zeros(m, d, dtype=torch.float64, device="cuda")

    def expert(rows, gate, up, down):
        a = x[rows]
        hid = _silu(a @ dequantize(fmt, gate, h, d).t()) * (a @ dequantize(fmt, up, h, d).t())
        return hid @ dequantize(fmt, down, d, h).t()

    per = t["gate"].shape[0] // e
    used = (route != 0).any(0).cpu().tolist()
    for i in range(e):
        if used[i]:
            rows = route[:, i].nonzero()[:, 0]
            at = slice(i * per, (i + 1) * per)
            y[rows] += route[rows, i, None] * expert(rows, t["gate"][at], t["up"][at], t["down"][at])
    if case["shared"]:
        every = torch.arange(m, device="cuda")
        gate = x @ t["sg"].double().t()
        y += 0.5 * (torch.tanh(gate / 2) + 1.0) * expert(every, t["gs"], t["us"], t["ds"])
    return {"y": y, "route": route}


def _exact_decode(case, g, seed):
    t, fmt = _decode_inputs(case, g), case["fmt"]
    d, ffn, nq, nkv = case["d"], case["ffn"], case["q_heads"], case["kv_heads"]
    hd, ctx, vocab = case["head_dim"], case["ctx"], case["vocab"]
    half = hd // 2

    def norm(v, w):
        return v / torch.sqrt((v * v).mean() + 1e-5) * w.double()

    def proj(b, rows, cols, v):
        return dequantize(fmt, b, rows, cols) @ v

    angle = ctx * torch.exp(-2.0 * torch.arange(half, dtype=torch.float64, device="cuda") / hd * math.log(500000.0))
    cos, sin = torch.cos(angle), torch.sin(angle)

    def rotate(v):
        a, b = v[:, :half], v[:, half:]
        return torch.cat((a * cos - b * sin, a * sin + b * cos), 1)

    x = t["embed"][int(seed) % vocab].double()
    out = {}
    for i, layer in enumerate(t["layers"]):
        qkv = proj(layer["qkv"], (nq + 2 * nkv) * hd, d, norm(x, layer["attn_norm"])).reshape(-1, hd)
        q = rotate(qkv[:nq]).reshape(nkv, nq // nkv, hd)
        k, v = rotate(qkv[nq:nq + nkv]).half(), qkv[nq + nkv:].half()
        out["k%d" % i], out["v%d" % i] = k.double(), v.double()
        keys = torch.cat((layer["k"], k[:, None]), 1).double()
        values = torch.cat((layer["v"], v[:, None]), 1).double()
        p = torch.softmax(q @ keys.transpose(1, 2).contiguous() / math.sqrt(hd), 2)
        x = x + proj(layer["o"], d, d, (p @ values).reshape(-1))
        n = norm(x, layer["ffn_norm"])
        hid = _silu(proj(layer["gate"], ffn, d, n)) * proj(layer["up"], ffn, d, n)
        x = x + proj(layer["down"], d, ffn, hid)
    logits = dequantize(case["head"], t["head"], vocab, d) @ norm(x, t["out_norm"])
    out.update(logits=logits, token=None)
    return out


def exact(case, seed):
    g, kind = _gen(seed), case["kind"]
    if kind in ("product", "int8"):
        b = blocks(case["fmt"], case["rows"], case["cols"], g)
        x = _x(case["m"], case["cols"], case.get("x", "f32"), g)
        x = _records(x, case["step"]) if kind == "int8" else x.double()
        return x @ dequantize(case["fmt"], b, case["rows"], case["cols"]).t()
    return _exact_moe(case, g) if kind == "moe" else _exact_decode(case, g, seed)
