"""What is timed and compared: the decode matmul and the layers around it, through the package's public entry points.

A case is one kind of call a serving program makes, at one size:

- linear:  dense_reader.linear.linear / matmul of one packed weight (bfloat8_b, bfloat4_b, bfloat16), from one row
           (decode) over a few (batched decode, verification of drafted tokens) to thousands (prefill), with column
           scales, a residual or the float32 output where a layer has them;
- glu:     the gated MLP's first half, gate and up weights apart, swiglu or geglu, with or without column scales;
- blocks:  a block list, several projections of one activation in one launch (Q, K, V and friends);
- int4:    the group-scaled W4A16 weight, one token or many rows;
- head:    the LM head, to token ids on the device (DeviceHead), or to the best candidates (records, then the merge);
- moe:     a mixture-of-experts layer: one token (router and gate/up in one launch, then down), or the rows of a batch;
- pack:    a weight's way in and out of the packed layout (loading a model, reading a weight back).

Weights are N(0, 0.02), activations standard normal with a few channels far larger, as transformer activations have;
column scales lie in 0.5 .. 1.5, group scales in 0.001 .. 0.011.
"""

import math
import random
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "tensix-kernels_amd"))
from common import device as dev  # noqa: E402
from dense_reader import linear  # noqa: E402
from int4 import w4a16  # noqa: E402
from lm_head_topk import lmhead  # noqa: E402
from moe import moe8  # noqa: E402

FORMATS = {"bfp8": linear.bfloat8_b, "bfp4": linear.bfloat4_b, "bf16": linear.bfloat16}
TILE_BYTES = {"bfp8": 1088, "bfp4": 576, "bf16": 2048, "int4": 576}  # a 32 x 32 tile of weights, exponents or scales in


def listed():
    return [
        # the smallest call a program makes (a small projection of one token): launch and host time count
        {"name": "decode_small", "kind": "linear", "fmt": "bfp8", "m": 1, "k": 1024, "n": 512, "opt": "none"},
        # one token through an MLP-sized bfloat8_b projection: the weight's bytes bound it
        {"name": "decode_row", "kind": "linear", "fmt": "bfp8", "m": 1, "k": 4096, "n": 14336, "opt": "none"},
        # one token through the gated MLP's gate and up, bfloat4_b with column scales
        {"name": "decode_glu", "kind": "glu", "fmt": "bfp4", "m": 1, "k": 4096, "n": 14336, "act": "swiglu",
         "scaled": True},
        # a batch of eight through the MLP's way down (a long K), the residual added in float32
        {"name": "batch_residual", "kind": "linear", "fmt": "bfp8", "m": 8, "k": 14336, "n": 4096, "opt": "residual32"},
        # a batch of 32: Q, K, V in bfloat8_b with column scales and O in bf16, one launch
        {"name": "batch_blocks", "kind": "blocks", "m": 32, "k": 4096,
         "blocks": "bfp8:4096:s bfp8:1024:s bfp8:1024:s bf16:4096:"},
        # prefill of a prompt of a thousand tokens through a scaled bfloat8_b projection
        {"name": "prefill_linear", "kind": "linear", "fmt": "bfp8", "m": 1000, "k": 4096, "n": 14336, "opt": "scale"},
        # prefill of a ragged prompt through the gated MLP's gate and up, bfloat4_b
        {"name": "prefill_glu", "kind": "glu", "fmt": "bfp4", "m": 333, "k": 4096, "n": 14336, "act": "swiglu",
         "scaled": False},
        # a batch of sixteen through an int4 weight with group scales
        {"name": "int4_rows", "kind": "int4", "m": 16, "k": 4096, "n": 14336},
        # the LM head of four sequences to token ids, rescored and picked on the device
        {"name": "lm_head", "kind": "head", "mode": "pick", "fmt": "bfp8", "m": 4, "k": 4096, "n": 128256},
        # one token through a mixture-of-experts layer of the gpt-oss-20b shape
        {"name": "moe_decode", "kind": "moe", "m": 1, "e": 32, "top": 4, "k": 2880, "n": 2880, "act": "swiglu_oai",
         "kblock": False},
        # 32 rows (a batch, or drafted tokens to verify) through the same layer
        {"name": "moe_rows", "kind": "moe", "m": 32, "e": 32, "top": 4, "k": 2880, "n": 2880, "act": "swiglu_oai",
         "kblock": False},
        # a projection's float weight packed at load time, and its held values read back
        {"name": "pack", "kind": "pack", "fmt": "bfp8", "k": 4096, "n": 14336, "src": "float32", "col_scale": False},
    ]


# --- drawn cases ------------------------------------------------------------------------------------------------------

MOST = 1000 * 4096 * 14336  # multiply-adds of the largest listed case


def _log(rng, lo, hi, step=1):
    """A whole number of lo .. hi, spread over its logarithm, a multiple of step."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(hi, max(lo, int(round(v / step)) * step)) // step * step


def _rows(rng, hi, k, n):
    """Rows 1 .. hi, as many as the largest listed case's work allows at k x n."""
    return max(1, min(_log(rng, 1, hi), MOST // (k * n)))


def draw(rng):
    kind = rng.choice(["linear"] * 5 + ["glu"] * 3 + ["blocks"] * 2 + ["int4"] * 2 + ["head", "moe", "moe", "pack"])
    fmt = rng.choice(["bfp8", "bfp4", "bf16"])
    k, n = _log(rng, 96, 14336, 32), _log(rng, 32, 14336)
    if kind == "linear":
        return {"kind": kind, "fmt": fmt, "m": _rows(rng, 2048, k, n), "k": k, "n": n,
                "opt": rng.choice(["none", "none", "scale", "scale32", "residual", "residual32", "out32"])}
    if kind == "glu":
        return {"kind": kind, "fmt": fmt, "m": _rows(rng, 1024, k, 2 * n), "k": k, "n": n,
                "act": rng.choice(["swiglu", "geglu"]), "scaled": rng.random() < 0.5}
    if kind == "blocks":
        parts = [f"{rng.choice(['bfp8', 'bfp4', 'bf16'])}:{_log(rng, 32, 4096, 32)}:{rng.choice(['s', ''])}"
                 for _ in range(rng.randint(2, 4))]
        return {"kind": kind, "m": _log(rng, 1, 32), "k": k, "blocks": " ".join(parts)}
    if kind == "int4":
        return {"kind": kind, "m": _rows(rng, 512, k, n), "k": k, "n": n}
    if kind == "head":
        return {"kind": kind, "mode": rng.choice(["pick", "merge"]), "fmt": fmt, "m": _log(rng, 1, 16),
                "k": _log(rng, 512, 4096, 32), "n": _log(rng, 4096, 128256, 32)}
    if kind == "moe":
        e = rng.choice([8, 16, 32, 64]) if rng.random() < 0.5 else 32
        k, n = _log(rng, 256, 2880, 32), _log(rng, 128, 2880, 32)
        while e * k * n > 32 * 2880 * 2880:
            k, n = max(256, k // 64 * 32), max(128, n // 64 * 32)
        return {"kind": kind, "m": _log(rng, 1, 32), "e": 32 * -(-e // 32), "top": rng.randint(1, 8), "k": k, "n": n,
                "act": rng.choice(["silu", "gelu_tanh", "swiglu_oai"]), "kblock": rng.random() < 0.3}
    return {"kind": kind, "fmt": fmt, "k": k, "n": n, "src": rng.choice(["float32", "bfloat16"]),
            "col_scale": rng.random() < 0.5}


# --- inputs -----------------------------------------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _weight(g, n, k):
    return torch.randn(n, k, generator=g, device="cuda") * 0.02


def _x(g, m, k):
    x = torch.randn(m, k, generator=g, device="cuda")
    x[:, torch.randint(0, k, (4,), generator=g, device="cuda")] *= 8.0
    return x.to(torch.bfloat16)


def _scales(g, n):
    return torch.rand(n, generator=g, device="cuda") + 0.5


def _x4(x):
    return x.reshape(1, 1, *x.shape)


def _block_spec(case):
    """[(format, columns, scaled)] of a blocks case."""
    return [(f, int(c), s == "s") for f, c, s in (b.split(":") for b in case["blocks"].split())]


def _floats(case, seed):
    """The float values a case is made of (the packed weights' sources among them), from the seed alone."""
    g, kind, k = _gen(seed), case["kind"], case["k"]
    f = {}
    if kind in ("linear", "glu", "int4", "head"):
        f["x"] = _x(g, case["m"], k)
    if kind == "linear":
        f["w"] = _weight(g, case["n"], k)
        if case["opt"].startswith("scale"):
            f["s"] = _scales(g, case["n"])
        if case["opt"].startswith("residual"):
            f["res"] = torch.randn(case["m"], case["n"], generator=g, device="cuda").to(torch.bfloat16)
    elif kind == "glu":
        f["gate"], f["up"] = _weight(g, case["n"], k), _weight(g, case["n"], k)
        if case["scaled"]:
            f["sg"], f["su"] = _scales(g, case["n"]), _scales(g, case["n"])
    elif kind == "blocks":
        f["x"] = _x(g, case["m"], k)
        f["blocks"] = [(fmt, _weight(g, n, k), _scales(g, n) if s else None) for fmt, n, s in _block_spec(case)]
    elif kind == "int4":
        f["codes"] = torch.randint(-7, 8, (case["n"], k), generator=g, device="cuda", dtype=torch.int8)
        f["s"] = (torch.rand(case["n"], k // 32, generator=g, device="cuda") * 0.01 + 0.001).to(torch.bfloat16)
    elif kind == "head":
        f["w"] = _weight(g, case["n"], k)
    elif kind == "moe":
        e, n = case["e"], case["n"]
        f["x"] = torch.randn(case["m"], k, generator=g, device="cuda").to(torch.bfloat16)
        f["logits"] = torch.randn(case["m"], e, generator=g, device="cuda") * 2
        f["bias"] = torch.randn(e, 2 * n, generator=g, device="cuda") * 0.1
        f["gate_up"] = torch.randn(e, k, 2 * n, generator=g, device="cuda") * 0.02
        f["down"] = torch.randn(e, n, k, generator=g, device="cuda") * 0.02
    else:
        f["w"] = _weight(g, case["n"], k).to(getattr(torch, case["src"]))
    return f


def prepare(case, seed):
    f, kind, d = _floats(case, seed), case["kind"], dev.open_device(0)
    s = {"case": case, "device": d}
    if kind == "linear":
        s["x"], s["w"] = _x4(f["x"]), linear.native_weight(d, f["w"], FORMATS[case["fmt"]])[0]
        dt = linear.float32 if case["opt"] == "scale32" else linear.bfloat16
        s["scale"] = linear.scale_tensor(d, f["s"], dtype=dt) if "s" in f else None
        s["res"] = _x4(f["res"]) if "res" in f else None
    elif kind == "glu":
        s["x"] = _x4(f["x"])
        s["w"] = tuple(linear.native_weight(d, f[p], FORMATS[case["fmt"]])[0] for p in ("gate", "up"))
        s["scale"] = tuple(linear.scale_tensor(d, f[p], dtype=linear.float32) if p in f else None for p in ("sg", "su"))
    elif kind == "blocks":
        s["x"], s["w"], c0 = _x4(f["x"]), [], 0
        for fmt, w, sc in f["blocks"]:
            pw = linear.native_weight(d, w, FORMATS[fmt])[0]
            s["w"].append((pw, c0) if sc is None else (pw, c0, linear.scale_tensor(d, sc, dtype=linear.float32)))
            c0 += w.shape[0] // 32
    elif kind == "int4":
        s["x"], s["w"], s["scale"] = f["x"], w4a16.int4_weight(d, f["codes"]), w4a16.group_scales(d, f["s"])
    elif kind == "head":
        s["x"] = _x4(f["x"])
        if case["mode"] == "pick":
            s["head"] = lmhead.DeviceHead(d, f["w"], fmt=case["fmt"], chunks=1, k=8, top=16, device_pick=True)
        else:
            s["w"] = linear.native_weight(d, f["w"], FORMATS[case["fmt"]])[0]
            s["records"] = linear.topk_result(d, linear.topk_slots(case["n"], 0), case["m"], 8)
            s["y"] = torch.empty(1, 1, case["m"], case["n"], dtype=torch.bfloat16, device="cuda")
    elif kind == "moe":
        m, top = case["m"], case["top"]
        s["x"], s["logits"] = _x4(f["x"]), _x4(f["logits"])
        s["p"] = moe8.pack(d, f["gate_up"], f["down"], gu_bias=f["bias"], kblock=case["kblock"])
        s["ids"] = torch.zeros(1, 1, m, top, dtype=torch.int16, device="cuda")
        s["wts"] = torch.zeros(1, 1, m, top, dtype=torch.bfloat16, device="cuda")
    else:
        s["w"] = f["w"]
    return s


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    if kind == "linear":
        o = {}
        if case["opt"].startswith("residual"):
            o["residual"] = s["res"]
        if case["opt"] in ("residual32", "out32"):
            o["out_dtype"] = linear.float32
        return linear.linear(s["x"], s["w"], s["scale"], **o)
    if kind == "glu":
        return linear.linear(s["x"], s["w"], s["scale"][0], activation=case["act"], scale_up=s["scale"][1])
    if kind == "blocks":
        return linear.linear(s["x"], s["w"], None)
    if kind == "int4":
        if case["m"] == 1:
            return w4a16.w4a16_linear(s["x"].reshape(1, 1, 1, -1), s["w"], s["scale"])
        return w4a16.rows_matmul(s["x"], s["w"], s["scale"])
    if kind == "head":
        m = case["m"]
        if case["mode"] == "pick":
            records = s["head"].logits_topk(s["x"], m)
            return {"records": records, "page": s["head"].picks[m]}
        spec = {"r": s["records"], "k": 8, "rows": m, "slot0": 0, "base": 0, "n": case["n"], "write_y": False,
                "fp32": True, "slots": 0}
        linear.matmul(s["x"], s["w"], None, out=s["y"], topk=spec)
        vals, ids = linear.topk_merge(s["records"], m, 8, k_out=32, fp32=True)
        return {"values": vals, "ids": ids}
    if kind == "moe":
        m, top, p, ids, wts = case["m"], case["top"], s["p"], s["ids"], s["wts"]
        if m == 1:
            h = moe8.route_gate_up(s["logits"], s["x"], p, ids, wts, top, act=case["act"], loaders=2)
            y = moe8.down(h, p, ids, top)
        else:
            moe8.route(s["logits"], ids, wts, top)
            h = moe8.gate_up_rows(s["x"], p, ids, wts, top, m, act=case["act"], loaders=2)
            y = moe8.down_rows(h, p, ids, top, m)
        return {"y": y, "h": h, "ids": ids, "weights": wts}
    w, scale = linear.native_weight(s["device"], s["w"], FORMATS[case["fmt"]], col_scale=case["col_scale"])
    out = {"codes": w.codes, "scale": scale, "held": linear.to_torch(w)}
    if w.exps is not None:
        out["exps"] = w.exps
    return out


# --- what a pass cannot do without ------------------------------------------------------------------------------------


def _wbytes(fmt, k, n):
    return k * n * TILE_BYTES[fmt] / 1024


def work(case):
    kind, k, m = case["kind"], case["k"], case.get("m", 0)
    if kind == "linear":
        n, opt = case["n"], case["opt"]
        b = _wbytes(case["fmt"], k, n) + 2 * m * k + m * n * (4 if opt in ("residual32", "out32") else 2)
        b += {"scale": 2 * n, "scale32": 4 * n, "residual": 2 * m * n, "residual32": 2 * m * n}.get(opt, 0)
        return {"bytes": b, "flops": 2 * m * k * n}
    if kind == "glu":
        n = case["n"]
        b = 2 * _wbytes(case["fmt"], k, n) + 2 * m * k + 2 * m * n + (8 * n if case["scaled"] else 0)
        return {"bytes": b, "flops": 4 * m * k * n}
    if kind == "blocks":
        spec = _block_spec(case)
        n = sum(c for _, c, _ in spec)
        b = sum(_wbytes(f, k, c) + (4 * c if s else 0) for f, c, s in spec) + 2 * m * k + 2 * m * n
        return {"bytes": b, "flops": 2 * m * k * n}
    if kind == "int4":
        n = case["n"]
        return {"bytes": _wbytes("int4", k, n) + 2 * m * k + 2 * m * n, "flops": 2 * m * k * n}
    if kind == "head":
        n = case["n"]
        return {"bytes": _wbytes(case["fmt"], k, n) + 2 * m * k + 128 * m, "flops": 2 * m * k * n}
    if kind == "moe":
        n, top, e = case["n"], case["top"], case["e"]
        chosen = e * (1 - (1 - top / e) ** m)  # experts of the rows' union, expected
        b = chosen * 3 * _wbytes("bfp4", k, n) + 2 * m * (2 * k + top * n)
        return {"bytes": b, "flops": 6 * m * top * k * n}
    n = case["n"]
    src = 4 if case["src"] == "float32" else 2
    return {"bytes": k * n * (src + 4) + 2 * _wbytes(case["fmt"], k, n), "flops": 0}


# --- the results in 64 bits -------------------------------------------------------------------------------------------

MANTISSA = {"bfp8": 7, "bfp4": 3}


def _pow2(e):
    """2^e in float64, from its bits."""
    return ((e.to(torch.int64) + 1023) << 52).view(torch.float64)


def _block_float(v, bits):
    """v [..., 16] float64 rounded to a block float: the exponent of the largest of the 16 shared, each value's 24-bit
    significand cut at the shared exponent's, rounded to `bits` bits half to even, at most 2^bits - 1."""
    e = torch.frexp(v.abs().amax(-1, keepdim=True)).exponent - 1  # 2^e <= max < 2^(e + 1)
    cut = torch.floor(v.abs() * _pow2(23 - e))
    q = torch.round(cut * 2.0 ** (bits - 24)).clamp(max=2**bits - 1)
    return q * v.sign() * _pow2(e - (bits - 1))


def _held(w, fmt, along_k=False):
    """[K, N] float64: the values a packed weight of w [N, K] holds (16 columns, or 16 k, share an exponent)."""
    if fmt == "bf16":
        return w.to(torch.bfloat16).double().t()
    v = (w if along_k else w.t()).double()
    c = v.shape[-1]
    v = torch.nn.functional.pad(v, (0, -c % 16)) if c % 16 else v
    h = _block_float(v.reshape(v.shape[0], -1, 16), MANTISSA[fmt]).reshape(v.shape)[:, :c]
    return h.t() if along_k else h


def _act(g, u, act):
    if act == "swiglu_oai":
        gc = g.clamp(max=7.0)
        return gc * torch.sigmoid(1.702 * gc) * (u.clamp(-7.0, 7.0) + 1)
    if act in ("geglu", "gelu_tanh"):
        return torch.nn.functional.gelu(g, approximate="tanh") * u
    return g * torch.sigmoid(g) * u


def _exact_moe(case, f):
    m, top, n, k = case["m"], case["top"], case["n"], case["k"]
    val, ids = torch.sort(f["logits"].double(), dim=1, descending=True, stable=True)
    ids, wts = ids[:, :top], torch.softmax(val[:, :top], dim=1)
    union = sorted(set(ids.flatten().tolist()))
    x, bias = f["x"].double(), f["bias"].to(torch.bfloat16).double()
    cols = top if m == 1 else min(case["e"], m * top)
    h = torch.zeros(1 if m == 1 else 32, cols, n, dtype=torch.float64, device="cuda")
    y = torch.zeros(1 if m == 1 else 32, k, dtype=torch.float64, device="cuda")
    for q, e in enumerate(union):
        def held(w):  # a [K, N] matrix of the expert
            return _held(w.t(), "bfp4", along_k=case["kblock"])

        up, gate = held(f["gate_up"][e, :, :n]), held(f["gate_up"][e, :, n:])
        we = (wts * (ids == e)).sum(1)  # the rows' weights of this expert
        he = _act(x @ gate + bias[e, n:], x @ up + bias[e, :n], case["act"]) * we[:, None]
        slot = int((ids[0] == e).nonzero()) if m == 1 else q
        h[:m, slot] = he
        y[:m] += he @ held(f["down"][e])
    shape = (1, 1, h.shape[0])
    return {"y": y.reshape(*shape, k), "h": h.reshape(*shape, cols * n), "ids": None,
            "weights": wts.reshape(1, 1, m, top)}


def exact(case, seed):
    f, kind = _floats(case, seed), case["kind"]
    if kind == "linear":
        y = f["x"].double() @ _held(f["w"], case["fmt"])
        if "s" in f:
            y = y * (f["s"] if case["opt"] == "scale32" else f["s"].to(torch.bfloat16)).double()
        return _x4(y + f["res"].double() if "res" in f else y)
    if kind == "glu":
        g, u = (f["x"].double() @ _held(f[p], case["fmt"]) for p in ("gate", "up"))
        if case["scaled"]:
            g, u = g * f["sg"].double(), u * f["su"].double()
        return _x4(_act(g, u, case["act"]))
    if kind == "blocks":
        cols = [f["x"].double() @ _held(w, fmt) * (1.0 if s is None else s.double()) for fmt, w, s in f["blocks"]]
        return _x4(torch.cat(cols, 1))
    if kind == "int4":
        y = f["x"].double() @ (f["codes"].double() * f["s"].double().repeat_interleave(32, dim=1)).t()
        return y.reshape(1, 1, 1, -1) if case["m"] == 1 else y
    if kind == "head":
        if case["mode"] == "pick":
            return None  # (keys, ids and counts: no computed numbers)
        y = f["x"].double() @ _held(f["w"], case["fmt"])
        m, n = y.shape
        tiles = torch.nn.functional.pad(y, (0, -n % 32), value=-math.inf).reshape(m, -1, 32)
        best = tiles.topk(8, dim=2).values.reshape(m, -1)
        return {"values": best.topk(32, dim=1).values, "ids": None}
    if kind == "moe":
        return _exact_moe(case, f)
    w = f["w"].float()
    c = torch.ones(case["n"], device="cuda")
    if case["col_scale"]:
        top = w.abs().amax(1).clamp(min=1e-8)
        c = top.to(torch.bfloat16).float()
        c = torch.where(c >= top, c, (c.view(torch.int32) + 0x10000).view(torch.float32))  # (the next bf16 up)
        w = w / c[:, None]
    held = _held(w, case["fmt"])
    held = torch.nn.functional.pad(held, (0, -held.shape[1] % 256))  # (columns padded over the device's eight banks)
    out = {"codes": None, "scale": c.double().reshape(1, 1, 1, -1), "held": _x4(held)}
    if case["fmt"] != "bf16":
        out["exps"] = None
    return out


def tolerance(case):
    kind = case["kind"]
    if kind == "pack":
        return "exact"
    if kind == "linear" and case["opt"] in ("residual32", "out32"):
        return {"rel": 1e-5, "max": 1e-4}
    if kind == "head":
        if case["mode"] == "pick":
            return {"rel": 0.0, "differ": 5e-3}  # (bf16 keys a rounding apart, and the ids behind them)
        return {"rel": 1e-5, "max": 1e-4, "differ": 5e-3}
    if kind == "moe":
        return {"rel": 1.2e-2, "max": 0.1}  # (the hidden values rounded to bf16 between the two halves)
    return {"rel": 7e-3, "max": 0.05}  # (one rounding to bf16)


if __name__ == "__main__":
    for c in listed() + [draw(random.Random(i)) for i in range(8)]:
        print(c, work(c))
