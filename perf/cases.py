"""The work this framework's users have it do, as cases that can be timed.

Every case goes through the public entry points: the device launchers of
``dianoia_amd.device`` for callers that keep tensors in HBM, and the
``lab_gpu_*`` command buffer (``dianoia_amd.forward``) for whole passes.
Shapes are those of ``bench.py`` and the tests, or generic ones; ``draw``
spreads each kind over the sizes, formats and options it is used with.

``exact`` states each result in 64 bits: the products of the quantized
operands (quantizing an input is part of the function, so its integers and
scales are formed as the format defines them), summed in float64.
"""

from __future__ import annotations

import dataclasses
import math

import numpy as np
import torch

from dianoia_amd import device as D
from dianoia_amd import forward as F

EPS = 1e-6


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # The smallest call: one decode projection of a small Q8 layer.
        {"name": "decode projection q8", "kind": "gemv", "fmt": "q8", "rows": 3072, "cols": 1024,
         "n": 1, "int8": True},
        # A decoder's MLP for one token: gate and up with their glue, then down.
        {"name": "decode mlp q4", "kind": "decode_mlp", "fmt": "q4", "hidden": 2048,
         "inter": 6144, "n": 1},
        # The greedy token: the Q8 LM head with its argmax.
        {"name": "lm head greedy q8", "kind": "lm_head", "rows": 151936, "cols": 2048},
        # One token's attention over a long context.
        {"name": "decode attention 4k", "kind": "attention", "n": 1, "position": 4095,
         "heads": 32, "kv_heads": 8, "hd": 128, "window": 0, "gate": False},
        # A prompt chunk (64 tokens, the largest the decoder takes at once)
        # through a norm and its Q4 MLP on prepacked weights.
        {"name": "prompt chunk mlp q4", "kind": "chunk_mlp", "hidden": 2048, "inter": 6144,
         "n": 64},
        # A long prompt's Q4 projection, 512 tokens at once, prepacked.
        {"name": "prefill product q4", "kind": "prefill_q4", "rows": 6144, "cols": 2048,
         "n": 512},
        # Causal attention of a 512-token prompt over its own keys.
        {"name": "prefill attention 512", "kind": "attention", "n": 512, "position": 0,
         "heads": 32, "kv_heads": 8, "hd": 128, "window": 0, "gate": False},
        # The vision encoder's MLP over 1024 patches; 4304 is not a multiple
        # of the 32-value block.
        {"name": "vision mlp q8", "kind": "vision_mlp", "hidden": 1152, "inter": 4304, "n": 1024},
        # A prompt chunk's projection of a Q8 model, weights as uploaded.
        {"name": "prompt chunk product q8", "kind": "batch", "fmt": "q8", "rows": 3072,
         "cols": 1024, "n": 64, "int8": True},
        # The vision projector with float inputs (mode 0, no quantization).
        {"name": "float product q8", "kind": "batch", "fmt": "q8", "rows": 4096, "cols": 4096,
         "n": 256, "int8": False},
        # Loading: a GGUF model's tied Q6_K embedding into the engine's Q8.
        {"name": "load q6k embedding", "kind": "load", "what": "q6k", "rows": 151936,
         "cols": 2048},
        # A whole pass through the command buffer: a 64-token prompt chunk
        # after 256 cached positions, then one token with its logits.
        {"name": "chunk and token", "kind": "model", "layers": "FFFFFF", "hidden": 2048,
         "inter": 6144, "heads": 16, "kv_heads": 8, "hd": 128, "vocab": 151936, "n": 64,
         "position": 256, "max_seq": 512, "window": 0, "sandwich": False, "gate": False},
    ]


def _log(rng, low, high, step=1):
    """A size between low and high, even over its logarithm, a multiple of step."""
    v = math.exp(rng.uniform(math.log(low), math.log(high)))
    return min(high, max(low, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(["gemv", "decode_mlp", "lm_head", "attention", "attention", "chunk_mlp",
                       "prefill_q4", "vision_mlp", "batch", "batch", "load", "model"])
    if kind == "gemv":
        return {"kind": kind, "fmt": rng.choice(["q8", "q4"]), "rows": _log(rng, 200, 16000),
                "cols": _log(rng, 256, 8192, 32), "n": rng.randint(1, 4),
                "int8": rng.random() < 0.75}
    if kind == "decode_mlp":
        return {"kind": kind, "fmt": rng.choice(["q8", "q4"]),
                "hidden": _log(rng, 512, 4096, 32), "inter": _log(rng, 1024, 12288, 32),
                "n": rng.randint(1, 4)}
    if kind == "lm_head":
        return {"kind": kind, "rows": _log(rng, 16001, 151936), "cols": _log(rng, 512, 2048, 32)}
    if kind == "attention":
        kv = rng.choice([2, 4, 8])
        n = 1 if rng.random() < 0.5 else _log(rng, 8, 1024)
        return {"kind": kind, "n": n,
                "position": _log(rng, 1, 16384) if n == 1 else _log(rng, 1, 4096) - 1,
                "heads": kv * rng.choice([1, 2, 4]), "kv_heads": kv,
                "hd": rng.choice([64, 128]), "window": rng.choice([0, 0, 0, 512]),
                "gate": rng.random() < 0.3}
    if kind == "chunk_mlp":
        return {"kind": kind, "hidden": _log(rng, 512, 4096, 32),
                "inter": _log(rng, 1024, 12288, 32), "n": rng.randint(5, 64)}
    if kind == "prefill_q4":
        return {"kind": kind, "rows": _log(rng, 768, 12288), "cols": _log(rng, 512, 4096, 32),
                "n": _log(rng, 65, 1024)}
    if kind == "vision_mlp":
        return {"kind": kind, "hidden": _log(rng, 512, 1536, 32), "inter": _log(rng, 1024, 6144),
                "n": _log(rng, 196, 2048)}
    if kind == "batch":
        return {"kind": kind, "fmt": rng.choice(["q8", "q4"]), "rows": _log(rng, 512, 8192),
                "cols": _log(rng, 512, 4096, 32), "n": _log(rng, 5, 1024),
                "int8": rng.random() < 0.5}
    if kind == "load":
        return {"kind": kind,
                "what": rng.choice(["q6k", "bf16_q8", "bf16_q4", "split_q8", "split_q4"]),
                "rows": _log(rng, 1000, 65536), "cols": _log(rng, 512, 4096, 256)}
    hd = rng.choice([64, 128])
    kv = rng.choice([1, 2, 4])
    return {"kind": "model", "layers": rng.choice(["CFCS", "FFF", "CCF", "FSFS"]),
            "hidden": rng.choice([512, 768, 1024]), "inter": _log(rng, 1024, 4096, 32),
            "heads": kv * rng.choice([1, 2, 4]), "kv_heads": kv, "hd": hd,
            "vocab": _log(rng, 1000, 32000), "n": rng.randint(2, 64),
            "position": _log(rng, 1, 1000), "max_seq": 1088, "window": 128,
            "sandwich": rng.random() < 0.5, "gate": rng.random() < 0.5}


# --------------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _q8(g, rows, cols):
    """Q8 weights: int8 in [-127, 127], fp32 block scales that fp16 holds."""
    qs = torch.randint(-127, 128, (rows, cols), dtype=torch.int8, device="cuda", generator=g)
    sc = torch.randn((rows, cols // 32), device="cuda", generator=g).abs().mul_(0.01)
    return qs, sc.half().float()


def _q4(g, rows, cols):
    """Q4 weights: two nibbles a byte, fp16 block scales (their bits)."""
    qs = torch.randint(0, 256, (rows, cols // 2), dtype=torch.uint8, device="cuda", generator=g)
    sc = torch.randn((rows, cols // 32), device="cuda", generator=g).abs().mul_(0.02)
    return qs, sc.half().view(torch.int16)


def _weights(fmt, g, rows, cols):
    return _q4(g, rows, cols) if fmt == "q4" else _q8(g, rows, cols)


def _x(g, *shape):
    return torch.randn(shape, device="cuda", generator=g)


def _out(*shape):
    return torch.empty(shape, device="cuda")


def _bytes(n):
    return torch.empty(n, dtype=torch.uint8, device="cuda")


def _pad32(n):
    return (n + 31) // 32 * 32


def _vision_weights(g, hidden, inter):
    """The two matrices of a vision MLP in bf16, as they lie in the file."""
    w1 = (torch.randn((inter, hidden), device="cuda", generator=g) * 0.02).bfloat16()
    w2 = (torch.randn((hidden, inter), device="cuda", generator=g) * 0.02).bfloat16()
    return w1, w2


def _load_source(g, what, rows, cols):
    if what.startswith("bf16"):
        return (torch.randn((rows, cols), device="cuda", generator=g) * 0.02).bfloat16()
    size = {"q6k": 210, "split_q8": 34, "split_q4": 18}[what]
    count = rows * cols // (256 if what == "q6k" else 32)
    blocks = torch.randint(0, 256, (count, size), dtype=torch.uint8, device="cuda", generator=g)
    d = (torch.randn(count, device="cuda", generator=g).abs().mul_(0.002) + 1e-4).half()
    at = 208 if what == "q6k" else 0
    blocks[:, at:at + 2] = d.view(torch.uint8).view(count, 2)
    return blocks


class _Model:
    """A decoder behind the command buffer, its cached positions filled; its
    GPU buffers go when the object does."""

    def __init__(self, case, seed):
        kinds = {"F": F.FULL, "S": F.SLIDING, "C": F.CONV}
        config = dataclasses.replace(
            F.qwen3_1_7b(), hidden=case["hidden"], intermediate=case["inter"],
            heads=case["heads"], kv_heads=case["kv_heads"], head_dim=case["hd"],
            vocab=case["vocab"], layer_types=[kinds[k] for k in case["layers"]],
            sliding_window=case["window"], sandwich=case["sandwich"], gate=case["gate"])
        self.fwd = F.GpuForward(config, max_seq=case["max_seq"], max_chunk=64, seed=seed)
        self.n, self.position = case["n"], case["position"]
        rng = np.random.default_rng(seed + 1)
        for block in self.fwd.state_blocks(self.position):
            block[:] = rng.standard_normal(len(block), dtype=np.float32)
        self.prompt = rng.standard_normal(self.n * config.hidden, dtype=np.float32)
        self.token = rng.standard_normal(config.hidden, dtype=np.float32)

    def __del__(self):
        if hasattr(self, "fwd"):
            self.fwd.dispose()

    def run(self):
        f = self.fwd
        f.reset()
        f.residual[:len(self.prompt)] = self.prompt
        f.forward(self.n, self.position)
        first = f.logits.copy()
        f.residual[:len(self.token)] = self.token
        f.forward(1, self.position + self.n)
        return {"chunk": first, "token": f.logits.copy()}


def prepare(case, seed):
    k, g = case["kind"], _gen(seed)
    s = {"case": case}
    if k == "gemv":
        s["w"] = _weights(case["fmt"], g, case["rows"], case["cols"])
        s["x"] = _x(g, case["n"], case["cols"])
        s["y"] = _out(case["n"], case["rows"])
    elif k == "decode_mlp":
        h, i, n = case["hidden"], case["inter"], case["n"]
        s["gate"], s["up"] = _weights(case["fmt"], g, i, h), _weights(case["fmt"], g, i, h)
        s["down"] = _weights(case["fmt"], g, h, i)
        s["x"], s["h"], s["y"] = _x(g, n, h), _out(n, i), _out(n, h)
    elif k == "lm_head":
        s["w"] = _q8(g, case["rows"], case["cols"])
        s["x"], s["y"] = _x(g, 1, case["cols"]), _out(case["rows"])
        s["token"] = torch.zeros(1, dtype=torch.int64, device="cuda")
        s["workspace"] = D.gemv_argmax_workspace()
    elif k == "attention":
        n, kv = case["n"], case["kv_heads"] * case["hd"]
        s["q"] = _x(g, n, case["heads"] * case["hd"])
        s["keys"], s["values"] = _x(g, case["position"] + n, kv), _x(g, case["position"] + n, kv)
        s["gate"] = _x(g, n, case["heads"]) if case["gate"] else None
        s["out"] = _out(n, case["heads"] * case["hd"])
    elif k == "chunk_mlp":
        h, i, n = case["hidden"], case["inter"], case["n"]
        for name, rows, cols in (("gate", i, h), ("up", i, h), ("down", h, i)):
            s[name] = _bytes(D.q4_f6pack_bytes(rows, cols))
            D.pack_q4_f6(*_q4(g, rows, cols), s[name], rows, cols)
        s["norm"] = torch.rand(h, device="cuda", generator=g) * 0.4 + 0.8
        s["x"], s["a"], s["y"] = _x(g, n, h), _out(n, h), _out(n, h)
        s["g"], s["u"] = _out(n, i), _out(n, i)
        s["pa"], s["ph"] = _bytes(D.f6_panel_bytes(n, h)), _bytes(D.f6_panel_bytes(n, i))
    elif k == "prefill_q4":
        rows, cols, n = case["rows"], case["cols"], case["n"]
        s["w"] = _bytes(D.q4_f6pack_bytes(rows, cols))
        D.pack_q4_f6(*_q4(g, rows, cols), s["w"], rows, cols)
        s["x"], s["y"] = _x(g, n, cols), _out(n, rows)
        s["panel"] = _bytes(D.f6_panel_bytes(n, cols))
    elif k == "vision_mlp":
        h, i, n = case["hidden"], case["inter"], case["n"]
        ip = _pad32(i)
        w1, w2 = _vision_weights(g, h, i)
        q1 = torch.zeros((ip, h), dtype=torch.int8, device="cuda")
        s1 = torch.zeros((ip, h // 32), device="cuda")
        q2, s2 = torch.empty((h, ip), dtype=torch.int8, device="cuda"), _out(h, ip // 32)
        D.quantize_q8_bf16(w1, q1, s1, i, h, h)
        D.quantize_q8_bf16(w2, q2, s2, h, i, ip)
        s["w1"], s["w2"] = _bytes(D.q8_i8pack_bytes(ip, h)), _bytes(D.q8_i8pack_bytes(h, ip))
        D.pack_q8_i8(q1, s1, s["w1"], ip, h)
        D.pack_q8_i8(q2, s2, s["w2"], h, ip)
        s["x"], s["h"], s["y"] = _x(g, n, h), _out(n, ip), _out(n, h)
        s["px"], s["ph"] = _bytes(D.i8_panel_bytes(n, h)), _bytes(D.i8_panel_bytes(n, ip))
    elif k == "batch":
        s["w"] = _weights(case["fmt"], g, case["rows"], case["cols"])
        s["x"] = _x(g, case["n"], case["cols"])
        s["y"] = _out(case["n"], case["rows"])
        s["workspace"] = D.matmul_workspace(case["cols"], case["n"])
    elif k == "load":
        rows, cols, what = case["rows"], case["cols"], case["what"]
        s["src"] = _load_source(g, what, rows, cols)
        if what.endswith("q4"):
            s["qs"] = torch.empty((rows, cols // 2), dtype=torch.uint8, device="cuda")
            s["scales"] = torch.empty((rows, cols // 32), dtype=torch.int16, device="cuda")
        else:
            s["qs"] = torch.empty((rows, cols), dtype=torch.int8, device="cuda")
            s["scales"] = _out(rows, cols // 32)
    else:
        s["model"] = _Model(case, seed)
    return s


def run(s):
    case = s["case"]
    k = case["kind"]
    if k == "gemv":
        f = {("q8", True): D.gemv_q8, ("q4", True): D.gemv_q4, ("q8", False): D.gemv_q8_float,
             ("q4", False): D.gemv_q4_float}[case["fmt"], case["int8"]]
        f(*s["w"], s["x"], s["y"], case["rows"], case["cols"], case["n"])
        return {"y": s["y"]}
    if k == "decode_mlp":
        q4 = case["fmt"] == "q4"
        (D.gate_up_q4 if q4 else D.gate_up_q8)(*s["gate"], *s["up"], s["x"], s["h"],
                                               case["inter"], case["hidden"], case["n"])
        (D.gemv_q4 if q4 else D.gemv_q8)(*s["down"], s["h"], s["y"], case["hidden"],
                                         case["inter"], case["n"])
        return {"h": s["h"], "y": s["y"]}
    if k == "lm_head":
        D.gemv_q8_argmax(*s["w"], s["x"], s["y"], s["token"], s["workspace"], case["rows"],
                         case["cols"])
        return {"logits": s["y"], "token": s["token"]}
    if k == "attention":
        D.attention(s["q"], s["keys"], s["values"], s["gate"], s["out"], case["position"],
                    case["n"], case["heads"], case["kv_heads"], case["hd"], case["window"])
        return {"out": s["out"]}
    if k == "chunk_mlp":
        h, i, n = case["hidden"], case["inter"], case["n"]
        D.rms_norm_f6panel(s["x"], s["norm"], s["a"], s["pa"], n, h, EPS)
        D.gemm_q4_f6s_multi([s["gate"], s["up"]], [s["g"], s["u"]], [i, i], s["pa"], h, n)
        D.swiglu_f6panel(s["g"], s["u"], s["ph"], n, i)
        D.gemm_q4_f6s(s["down"], s["ph"], s["y"], h, i, n)
        return {"a": s["a"], "h": s["g"], "y": s["y"]}
    if k == "prefill_q4":
        D.quantize_q8_f6panel(s["x"], s["panel"], case["n"], case["cols"])
        D.gemm_q4_f6p(s["w"], s["panel"], s["y"], case["rows"], case["cols"], case["n"])
        return {"y": s["y"]}
    if k == "vision_mlp":
        h, n = case["hidden"], case["n"]
        ip = _pad32(case["inter"])
        D.quantize_q8_i8panel(s["x"], s["px"], n, h)
        D.gemm_q8_i8p(s["w1"], s["px"], s["h"], ip, h, n)
        D.gelu(s["h"])
        D.quantize_q8_i8panel(s["h"], s["ph"], n, ip)
        D.gemm_q8_i8p(s["w2"], s["ph"], s["y"], h, ip, n)
        return {"h": s["h"], "y": s["y"]}
    if k == "batch":
        (D.matmul_q4 if case["fmt"] == "q4" else D.matmul_q8)(
            *s["w"], s["x"], s["y"], case["rows"], case["cols"], case["n"], case["int8"],
            s["workspace"])
        return {"y": s["y"]}
    if k == "load":
        rows, cols, what = case["rows"], case["cols"], case["what"]
        if what == "q6k":
            D.q6k_to_q8(s["src"], s["qs"], s["scales"], rows, cols)
        elif what == "bf16_q8":
            D.quantize_q8_bf16(s["src"], s["qs"], s["scales"], rows, cols, cols)
        elif what == "bf16_q4":
            D.quantize_q4_bf16(s["src"], s["qs"], s["scales"], rows, cols)
        else:
            (D.split_q8_0 if what == "split_q8" else D.split_q4_0)(
                s["src"], s["qs"], s["scales"], rows * cols // 32)
        return {"qs": s["qs"], "scales": s["scales"]}
    return s["model"].run()


# ----------------------------------------------------- what a pass cannot avoid

def _wbytes(fmt, rows, cols):
    return rows * (cols // 32) * (18 if fmt == "q4" else 36)


def _visible(case):
    """Query-key pairs of one head, and key rows that are read."""
    n, p, w = case["n"], case["position"], case["window"]
    pairs = sum(min(p + t + 1, w) if w else p + t + 1 for t in range(n))
    first = max(0, p - w + 1) if w else 0
    return pairs, p + n - first


def work(case):
    k, n = case["kind"], case.get("n", 1)
    if k in ("gemv", "batch", "prefill_q4", "lm_head"):
        rows, cols = case["rows"], case["cols"]
        fmt = case.get("fmt", "q4" if k == "prefill_q4" else "q8")
        return {"bytes": _wbytes(fmt, rows, cols) + 4 * n * (rows + cols),
                "flops": 2 * rows * cols * n}
    if k in ("decode_mlp", "chunk_mlp"):
        h, i = case["hidden"], case["inter"]
        return {"bytes": 3 * _wbytes(case.get("fmt", "q4"), i, h) + 4 * n * (2 * h + i)
                + (4 * n * h if k == "chunk_mlp" else 0), "flops": 6 * h * i * n}
    if k == "vision_mlp":
        h, i = case["hidden"], case["inter"]
        return {"bytes": 2 * _wbytes("q8", _pad32(i), h) + 4 * n * (2 * h + i),
                "flops": 4 * h * i * n}
    if k == "attention":
        pairs, rows = _visible(case)
        return {"bytes": 4 * (2 * rows * case["kv_heads"] + 2 * n * case["heads"]) * case["hd"],
                "flops": 4 * pairs * case["heads"] * case["hd"]}
    if k == "load":
        values = case["rows"] * case["cols"]
        into = 18 / 32 if case["what"].endswith("q4") else 36 / 32
        return {"bytes": int(values * (into + {"q6k": 210 / 256, "bf16_q8": 2, "bf16_q4": 2,
                                               "split_q8": 34 / 32, "split_q4": 18 / 32}
                                       [case["what"]])), "flops": 0}
    h, i, kv = case["hidden"], case["inter"], case["kv_heads"] * case["hd"]
    q = case["heads"] * case["hd"]
    per = {"C": 4 * h * h, "F": 2 * q * h + 2 * kv * h}
    per["S"] = per["F"]
    body = sum(per[c] + 3 * h * i for c in case["layers"])
    cached = sum(2 * kv * (case["position"] + n) for c in case["layers"] if c != "C")
    head = case["vocab"] * h
    return {"bytes": 2 * (body * 18 // 32 + head * 36 // 32) + 4 * (2 * cached + 2 * case["vocab"]),
            "flops": 2 * body * (n + 1) + 4 * head}


# Four times what was measured. A product, or an attention, summed in float32
# is 1e-7 to 3.5e-7 of its norm away from 64 bits. Where a result is quantized
# again, a value at a rounding boundary moves by one step of its block's 127:
# an MLP's second product then moves by up to 7e-5 of its norm. In a whole
# pass every layer adds to that: with its inputs moved by one unit in their
# last place, the logits of the 2048-wide decoder move by 1.4e-3, those of
# narrow ones with a norm after each block by up to 2e-2.
def tolerance(case):
    k = case["kind"]
    if k == "load":
        return "exact"
    if k == "decode_mlp":
        return {"rel": 1.5e-6, "max": 2e-5}
    if k in ("chunk_mlp", "vision_mlp"):
        return {"rel": 3e-4, "max": 0.01}
    if k == "model":
        return {"rel": 6e-3, "max": 0.03} if case["hidden"] >= 2048 else {"rel": 0.03, "max": 0.3}
    if k == "lm_head":
        return {"rel": 1.5e-6, "max": 2e-5, "differ": 0.0}
    return {"rel": 1.5e-6, "max": 2e-5}


# ------------------------------------------------------------ the same in 64 bits

def _quantize(x):
    """The engine's Q8 of float32 rows: (integers, float32 block scales)."""
    b = x.float().reshape(x.shape[0], -1, 32)
    amax = b.abs().amax(2, keepdim=True)
    scale = (amax.double() / 127.0).float()
    inv = torch.where(scale > 0, (1.0 / scale.double()).float(), torch.zeros_like(scale))
    t = b * inv
    t = t + torch.copysign(torch.full_like(t, 0.5), t)
    return t.clamp(-127, 127).trunc().reshape(x.shape[0], -1), scale[:, :, 0]


def _widen(q, scales):
    return (q.double().reshape(q.shape[0], -1, 32) * scales.double()[:, :, None]).reshape(
        q.shape[0], -1)


def _dense(fmt, w):
    """A weight matrix's values in float64."""
    qs, sc = w
    if fmt == "q8":
        return _widen(qs, sc)
    b = qs.reshape(qs.shape[0], -1, 16)
    q = torch.cat([(b & 15).to(torch.int8) - 8, (b >> 4).to(torch.int8) - 8], 2)
    return _widen(q.reshape(qs.shape[0], -1), sc.view(torch.float16))


def _product(fmt, w, x, int8=True):
    xv = _widen(*_quantize(x)) if int8 else x.double()
    parts = [xv @ _dense(fmt, (w[0][r:r + 16384], w[1][r:r + 16384])).T
             for r in range(0, w[0].shape[0], 16384)]
    return torch.cat(parts, 1)


def _silu(v):
    return v / (1 + torch.exp(-v))


def _gelu(v):
    """With the erf of Abramowitz and Stegun 7.1.26, as the encoder defines it."""
    z = v / 1.4142135623730951
    t = 1 / (1 + 0.3275911 * z.abs())
    poly = ((((1.061405429 * t - 1.453152027) * t + 1.421413741) * t - 0.284496736) * t
            + 0.254829592) * t
    erf = torch.copysign(1 - poly * torch.exp(-z * z), z)
    return 0.5 * v * (1 + erf)


def _attention(s, case):
    n, p, hd, w = case["n"], case["position"], case["hd"], case["window"]
    heads, group = case["heads"], case["heads"] // case["kv_heads"]
    q = s["q"].double().view(n, heads, hd)
    keys = s["keys"].double().view(p + n, -1, hd)
    values = s["values"].double().view(p + n, -1, hd)
    at = torch.arange(p + n, device="cuda")[None]
    own = torch.arange(p, p + n, device="cuda")[:, None]
    seen = (at <= own) & (at > own - w) if w else at <= own
    out = torch.empty((n, heads, hd), dtype=torch.float64, device="cuda")
    for h in range(heads):
        a = (q[:, h] @ keys[:, h // group].T / math.sqrt(hd)).masked_fill(~seen, -math.inf)
        out[:, h] = torch.softmax(a, 1) @ values[:, h // group]
    if s["gate"] is not None:
        out *= torch.sigmoid(s["gate"].double())[:, :, None]
    return out.view(n, heads * hd)


def exact(case, seed):
    k, g = case["kind"], _gen(seed)
    if k in ("load", "model"):
        return None
    if k == "attention":
        return {"out": _attention(prepare(case, seed), case)}
    if k in ("gemv", "batch"):
        w = _weights(case["fmt"], g, case["rows"], case["cols"])
        return {"y": _product(case["fmt"], w, _x(g, case["n"], case["cols"]), case["int8"])}
    if k == "lm_head":
        w = _q8(g, case["rows"], case["cols"])
        y = _product("q8", w, _x(g, 1, case["cols"]))[0]
        return {"logits": y, "token": y.argmax().reshape(1)}
    if k == "prefill_q4":
        w = _q4(g, case["rows"], case["cols"])
        return {"y": _product("q4", w, _x(g, case["n"], case["cols"]))}
    if k == "vision_mlp":
        h, i, n = case["hidden"], case["inter"], case["n"]
        w1, w2 = _vision_weights(g, h, i)
        pad = _pad32(i) - i
        q1 = _quantize(torch.nn.functional.pad(w1.float(), (0, 0, 0, pad)))
        q2 = _quantize(torch.nn.functional.pad(w2.float(), (0, pad)))
        a = _gelu(_product("q8", q1, _x(g, n, h)))
        return {"h": a, "y": _product("q8", q2, a)}
    h, i, n, fmt = case["hidden"], case["inter"], case["n"], case.get("fmt", "q4")
    gate, up, down = (_weights(fmt, g, r, c) for r, c in ((i, h), (i, h), (h, i)))
    if k == "decode_mlp":
        x = _x(g, n, h)
        a = _silu(_product(fmt, gate, x)) * _product(fmt, up, x)
        return {"h": a, "y": _product(fmt, down, a)}
    norm = torch.rand(h, device="cuda", generator=g) * 0.4 + 0.8
    x = _x(g, n, h).double()
    a = norm.double() * x / torch.sqrt(x.square().mean(1, keepdim=True) + EPS)
    b = _silu(_product(fmt, gate, a)) * _product(fmt, up, a)
    return {"a": a, "h": b, "y": _product(fmt, down, b)}
