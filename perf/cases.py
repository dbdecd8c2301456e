"""Performance cases of the quantised matmul library: what a program that runs
a Q4_0 / Q8_0 / FP16 language model asks of it, through hypno_amd's public
functions, from one 2048 x 2048 matrix-vector product to the feed-forward
block of a 2048-token prompt.

A case is a plain dict.  Its "kind" says what one pass does:

  gemv    one matmul_vec_auto: y = W x (+ bias) for one token
  decode  the projections of `layers` transformer layers for one token, four
          GemvPlans a layer: [q, k, v], [o], [gate, up], [down], with the RMS
          norms and silu(gate) * up as plan prologues
  mlp     the feed-forward block of `tokens` tokens: rms_norm, gate and up,
          silu_mul, down
  head    the vocabulary projection of `tokens` tokens
  sample  the next token from one row of logits
  codec   quantise an fp32 tensor and dequantise the blocks again
"""
import math

import numpy as np
import torch

import hypno_amd as hk

EPS = 1e-5
DTYPES = {"q4_0": hk.DType.Q4_0, "q8_0": hk.DType.Q8_0, "f16": hk.DType.FP16}
BLOCK_BYTES = {"q4_0": 18, "q8_0": 34, "f16": 64}  # of 32 weights


def listed():
    return [
        # The smallest call of the drop-in use: one 2048 x 2048 projection of a
        # one-token step, x and y in host memory, the weights registered once.
        {"name": "gemv_host_small", "kind": "gemv", "dtype": "q4_0", "n": 2048, "m": 2048,
         "bias": False, "host": True},
        # A one-token down projection whose row length (344 blocks) is no
        # power-of-two multiple of the wavefront, with a bias.
        {"name": "gemv_long_rows", "kind": "gemv", "dtype": "q4_0", "n": 4096, "m": 11008,
         "bias": True, "host": False},
        # A decode step: eight layers of a 7B model, one token.
        {"name": "decode_step", "kind": "decode", "layers": 8, "hidden": 4096, "kv": 1024,
         "ffn": 14336},
        # A few sequences decoded together.
        {"name": "mlp_few_tokens", "kind": "mlp", "dtype": "q4_0", "tokens": 8, "hidden": 4096,
         "ffn": 14336, "col": False},
        # A prompt of ordinary length on a 3B model.
        {"name": "mlp_prompt", "kind": "mlp", "dtype": "q4_0", "tokens": 512, "hidden": 3072,
         "ffn": 8192, "col": False},
        # The largest: a long prompt on a 7B model.
        {"name": "mlp_long_prompt", "kind": "mlp", "dtype": "q4_0", "tokens": 2048,
         "hidden": 4096, "ffn": 14336, "col": False},
        # Widths that are whole blocks but no multiples of 256 (2880 = 45 * 64,
        # 7200 = 225 * 32) and a token count that fills no tile.
        {"name": "mlp_ragged", "kind": "mlp", "dtype": "q4_0", "tokens": 333, "hidden": 2880,
         "ffn": 7200, "col": False},
        # A prompt on Q8_0 weights.
        {"name": "mlp_q8_0", "kind": "mlp", "dtype": "q8_0", "tokens": 512, "hidden": 4096,
         "ffn": 14336, "col": False},
        # A prompt on a model stored column-major.
        {"name": "mlp_col_major", "kind": "mlp", "dtype": "q4_0", "tokens": 128, "hidden": 2048,
         "ffn": 5632, "col": True},
        # The FP16 vocabulary projection of a one-token step.
        {"name": "head_f16", "kind": "head", "dtype": "f16", "tokens": 1, "vocab": 128256,
         "hidden": 4096},
        # Nucleus sampling over a full vocabulary.
        {"name": "sample_top_p", "kind": "sample", "vocab": 128256, "temperature": 1.0,
         "top_p": 0.9, "top_k": 0},
        # Weight conversion of one 4096 x 14336 tensor, and back.
        {"name": "codec_q4_0", "kind": "codec", "dtype": "q4_0", "elems": 4096 * 14336},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi, step=None):
    """A matrix width: most are multiples of 256, some of 64 or 32 only."""
    step = step or rng.choice([256, 256, 256, 64, 32])
    return min(hi // step * step, max(step, (_log(rng, lo, hi) + step // 2) // step * step))


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "decode", "mlp", "mlp", "mlp", "mlp", "head", "sample",
                       "codec"])
    dtype = rng.choice(["q4_0", "q4_0", "q8_0", "f16"])
    if kind == "gemv":
        m = _width(rng, 512, 16384)
        if rng.random() < 0.15:
            m += rng.randrange(1, 32)  # blocks that straddle rows
        return {"kind": kind, "dtype": dtype, "n": _log(rng, 256, 16384), "m": m,
                "bias": rng.random() < 0.5, "host": rng.random() < 0.25}
    if kind == "decode":
        hidden = _width(rng, 1024, 4096, 256)
        return {"kind": kind, "layers": rng.randrange(1, 9), "hidden": hidden,
                "kv": 128 * rng.randrange(1, 9), "ffn": _width(rng, 2048, 14336)}
    if kind == "mlp":
        if rng.random() < 0.25:  # column-major (Q4_0 only)
            return {"kind": kind, "dtype": "q4_0", "tokens": _log(rng, 1, 128),
                    "hidden": _width(rng, 512, 2048), "ffn": _width(rng, 1024, 5632),
                    "col": True}
        hidden, ffn = _width(rng, 512, 4096), _width(rng, 1024, 14336)
        tokens = _log(rng, 1, 2048)
        if hidden % 256 or ffn % 256:
            hidden, ffn, tokens = min(hidden, 2880), min(ffn, 7200), _log(rng, 1, 333)
        return {"kind": kind, "dtype": dtype, "tokens": tokens, "hidden": hidden, "ffn": ffn,
                "col": False}
    if kind == "head":
        return {"kind": kind, "dtype": dtype, "tokens": _log(rng, 1, 128),
                "vocab": _log(rng, 16000, 128256), "hidden": _width(rng, 1024, 4096, 256)}
    if kind == "sample":
        return {"kind": kind, "vocab": _log(rng, 4000, 152064),
                "temperature": rng.choice([0.0, 0.5, 0.7, 1.0, 1.3]),
                "top_p": rng.choice([0.5, 0.8, 0.9, 0.95, 1.0]),
                "top_k": rng.choice([0, 0, 20, 40, 200])}
    return {"kind": kind, "dtype": rng.choice(["q4_0", "q8_0"]),
            "elems": 32 * _log(rng, 1 << 10, 4096 * 14336 // 32) + rng.choice([0, 0, 17])}


# --- inputs ------------------------------------------------------------------------

def _gen(seed, what):
    return torch.Generator(device="cuda").manual_seed(seed * 1000 + what)


def _normal(seed, what, shape, std=1.0):
    return torch.randn(shape, generator=_gen(seed, what), device="cuda").mul_(std)


def _hidden(seed, what, tokens, width):
    """Hidden states: unit normal, with a few channels an order larger."""
    x = _normal(seed, what, (tokens, width))
    x[:, ::509] *= 10.0
    return x


def _norm_weight(seed, what, width):
    return _normal(seed, what, (width,), 0.1).add_(1.0)


def _round_half_away(v):
    return torch.trunc(v + torch.copysign(torch.full_like(v, 0.5), v))


def _scales(flat, dtype):
    """fp32 blocks [nb, 32] of a flat tensor, and each block's scale before it
    is rounded to fp16."""
    v = flat[: flat.numel() // 32 * 32].view(-1, 32)
    amax = v.abs().amax(dim=1, keepdim=True)
    s = amax / torch.tensor(7.0 if dtype == "q4_0" else 127.0, device="cuda")
    return v, torch.where(amax > 0, s, torch.ones_like(s))


def _pack(flat, dtype):
    """Q4_0 / Q8_0 block bytes, or FP16 bytes, of a flat fp32 tensor."""
    if dtype == "f16":
        return flat.half().view(torch.uint8)
    v, s = _scales(flat, dtype)
    d = s.half()
    out = torch.empty(v.shape[0], BLOCK_BYTES[dtype], dtype=torch.uint8, device="cuda")
    out[:, :2] = d.view(torch.uint8).view(-1, 2)
    if dtype == "q4_0":
        q = (_round_half_away(v / s).clamp_(-8, 7) + 8).to(torch.uint8)
        out[:, 2:] = q[:, 0::2] | (q[:, 1::2] << 4)
    else:
        out[:, 2:] = (_round_half_away(v / d.float()).clamp_(-127, 127) + 128).to(torch.uint8)
    return out.view(-1)


def _unpack(q, dtype, count):
    """The first `count` weights that packed bytes stand for, in 64 bits."""
    if dtype == "f16":
        return q.view(torch.float16).double()[:count]
    b = q.view(-1, BLOCK_BYTES[dtype])
    d = b[:, :2].contiguous().view(torch.float16).double()
    if dtype == "q4_0":
        n = torch.stack([b[:, 2:] & 15, b[:, 2:] >> 4], dim=2).view(-1, 32).double().sub_(8)
    else:
        n = b[:, 2:].double().sub_(128)
    return n.mul_(d).view(-1)[:count]


def _weights(seed, what, n, m, dtype):
    """A row-major [n][m] matrix, flattened and padded to whole blocks."""
    w = _normal(seed, what, (n * m + (-(n * m)) % 32,), 0.02)
    return _pack(w, dtype)


def _layer_shapes(case):
    h, kv, f = case["hidden"], case["kv"], case["ffn"]
    return [("q", h, h), ("k", kv, h), ("v", kv, h), ("o", h, h), ("gate", f, h), ("up", f, h),
            ("down", h, f)]


def _empty(*shape):
    return torch.empty(shape, dtype=torch.float32, device="cuda")


class _HostWeight:
    """A weight tensor in host memory, registered with the library."""

    def __init__(self, w):
        self.w = w.cpu().numpy()
        hk.register_weight(self.w)

    def __del__(self):
        hk.unregister_weight(self.w)


def _inputs(case, seed):
    """Everything a pass reads that is drawn from the seed, on the GPU."""
    kind = case["kind"]
    if kind == "gemv":
        n, m = case["n"], case["m"]
        return {"w": _weights(seed, 1, n, m, case["dtype"]), "x": _hidden(seed, 2, 1, m).view(-1),
                "bias": _normal(seed, 3, (n,)) if case["bias"] else None}
    if kind == "decode":
        layers = []
        for i in range(case["layers"]):
            t = {name: _weights(seed, 100 + 10 * i + j, n, m, "q4_0")
                 for j, (name, n, m) in enumerate(_layer_shapes(case))}
            t["attn_norm"] = _norm_weight(seed, 107 + 10 * i, case["hidden"])
            t["ffn_norm"] = _norm_weight(seed, 108 + 10 * i, case["hidden"])
            layers.append(t)
        return {"x": _hidden(seed, 1, 1, case["hidden"]).view(-1), "layers": layers}
    if kind == "mlp":
        h, f = case["hidden"], case["ffn"]
        up, down = ((h, f), (f, h)) if case["col"] else ((f, h), (h, f))
        return {"x": _hidden(seed, 1, case["tokens"], h), "norm": _norm_weight(seed, 2, h),
                "gate": _weights(seed, 3, *up, case["dtype"]),
                "up": _weights(seed, 4, *up, case["dtype"]),
                "down": _weights(seed, 5, *down, case["dtype"])}
    if kind == "head":
        return {"x": _hidden(seed, 1, case["tokens"], case["hidden"]),
                "w": _weights(seed, 2, case["vocab"], case["hidden"], case["dtype"])}
    if kind == "sample":
        return {"logits": _normal(seed, 1, (case["vocab"],), 3.0)}
    return {"data": _normal(seed, 1, (case["elems"],), 0.02)}


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    kind = case["kind"]
    if kind == "gemv":
        s["dtype"] = DTYPES[case["dtype"]]
        if case["host"]:
            s["keep"] = _HostWeight(s["w"])
            s["w"] = s["keep"].w
            s["x"] = s["x"].cpu().numpy()
            s["bias"] = None if s["bias"] is None else s["bias"].cpu().numpy()
            s["y"] = np.empty(case["n"], np.float32)
        else:
            s["y"] = _empty(case["n"])
    elif kind == "decode":
        s["plans"], s["kv"] = [], []
        shapes = {name: (n, m) for name, n, m in _layer_shapes(case)}
        x = s["x"]
        for t in s["layers"]:
            y = {name: _empty(n) for name, (n, m) in shapes.items()}

            def job(name, x, pro=None):
                j = (y[name], t[name], x, None, *shapes[name])
                return j if pro is None else j + (pro,)

            attn, ffn = ("rms_norm", t["attn_norm"], EPS), ("rms_norm", t["ffn_norm"], EPS)
            # (what attention makes of q, k and v is not this library's: o reads q)
            s["plans"] += [hk.GemvPlan([job("q", x, attn), job("k", x, attn), job("v", x, attn)]),
                           hk.GemvPlan([job("o", y["q"])]),
                           hk.GemvPlan([job("gate", y["o"], ffn), job("up", y["o"], ffn)]),
                           hk.GemvPlan([job("down", y["gate"], ("silu_mul", y["up"]))])]
            s["kv"].append((y["k"], y["v"]))
            x = y["down"]
        s["y"] = x
    elif kind == "mlp":
        s["dtype"] = DTYPES[case["dtype"]]
        t, h, f = case["tokens"], case["hidden"], case["ffn"]
        s["normed"], s["g"], s["u"], s["y"] = _empty(t, h), _empty(t, f), _empty(t, f), _empty(t, h)
    elif kind == "head":
        s["dtype"] = DTYPES[case["dtype"]]
        s["y"] = _empty(case["tokens"], case["vocab"])
    elif kind == "sample":
        s["rng"] = torch.tensor([seed * 7919 + 12345], dtype=torch.int64, device="cuda")
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "gemv":
        hk.matmul_vec_auto(s["y"], s["w"], s["dtype"], s["x"], s["bias"], case["n"], case["m"])
        return s["y"]
    if kind == "decode":
        for plan in s["plans"]:
            plan.run()
        return {"y": s["y"], "kv": s["kv"]}
    if kind == "mlp":
        t, h, f, dt, col = case["tokens"], case["hidden"], case["ffn"], s["dtype"], case["col"]
        hk.rms_norm(s["x"], s["norm"], EPS, rows=t, out=s["normed"])
        hk.batch_matmul(s["g"], s["gate"], dt, s["normed"], f, h, t, col_major=col)
        hk.batch_matmul(s["u"], s["up"], dt, s["normed"], f, h, t, col_major=col)
        hk.silu_mul(s["g"], s["u"], out=s["g"])
        hk.batch_matmul(s["y"], s["down"], dt, s["g"], h, f, t, col_major=col)
        return s["y"]
    if kind == "head":
        hk.batch_matmul(s["y"], s["w"], s["dtype"], s["x"], case["vocab"], case["hidden"],
                        case["tokens"])
        return s["y"]
    if kind == "sample":
        if case["temperature"] == 0.0:
            return {"token": hk.argmax(s["logits"])}
        token = hk.sample_token(s["logits"], case["temperature"], case["top_p"], case["top_k"],
                                s["rng"])
        return {"token": token, "rng": s["rng"]}
    if case["dtype"] == "q4_0":
        q = hk.quantize_f32_to_q4_0(s["data"])
        return {"q": q, "back": hk.dequantize_q4_0(q)}
    q = hk.quantize_f32_to_q8_0(s["data"])
    return {"q": q, "back": hk.dequantize_q8_0(q)}


# --- what a pass cannot do without, and how exact it is -------------------------------

def _weight_bytes(case, n, m):
    dtype = case.get("dtype", "q4_0")
    return 2 * n * m if dtype == "f16" else -(-(n * m) // 32) * BLOCK_BYTES[dtype]


def work(case):
    kind = case["kind"]
    if kind == "gemv":
        n, m = case["n"], case["m"]
        return {"bytes": _weight_bytes(case, n, m) + 4 * (m + n * (2 if case["bias"] else 1)),
                "flops": 2 * n * m}
    if kind == "decode":
        wb = sum(_weight_bytes(case, n, m) for _, n, m in _layer_shapes(case))
        weights = sum(n * m for _, n, m in _layer_shapes(case))
        h, kv = case["hidden"], case["kv"]
        return {"bytes": case["layers"] * (wb + 8 * h + 8 * kv) + 8 * h,
                "flops": 2 * case["layers"] * weights}
    if kind == "mlp":
        t, h, f = case["tokens"], case["hidden"], case["ffn"]
        return {"bytes": 3 * _weight_bytes(case, h, f) + 8 * t * h + 4 * h, "flops": 6 * t * h * f}
    if kind == "head":
        t, v, h = case["tokens"], case["vocab"], case["hidden"]
        return {"bytes": _weight_bytes(case, v, h) + 4 * t * (h + v), "flops": 2 * t * v * h}
    if kind == "sample":
        return {"bytes": 4 * case["vocab"], "flops": 3 * case["vocab"]}
    n = case["elems"]
    return {"bytes": 8 * n + n // 32 * BLOCK_BYTES[case["dtype"]], "flops": 3 * n}


def tolerance(case):
    kind = case["kind"]
    if kind in ("sample", "codec"):
        return "exact"  # the token, the generator's state and every byte are defined
    # Measured against exact(), times about four:
    if kind == "decode":
        return {"rel": 4e-4}  # 1e-4 after eight layers of 19-bit activations, fp32 sums
    if case.get("tokens", 1) < 16 or case.get("col"):
        if case.get("col") or case["dtype"] == "f16":
            return {"rel": 1e-5}  # fp32 sums
        return {"rel": 4e-5 if kind == "mlp" else 2e-5}  # 19-bit activations, fp32 sums
    # from 16 tokens activations are rounded to fp16, and Q8_0 weights once: 4-5e-4
    return {"rel": 2e-3}


def _rms_norm(x, weight):
    return x / (x.square().mean(dim=-1, keepdim=True) + EPS).sqrt() * weight


def exact(case, seed):
    kind = case["kind"]
    if kind == "sample":
        return None  # whole numbers
    s = _inputs(case, seed)
    dtype = case.get("dtype", "q4_0")

    def times(x, w, n, m, col=False):
        w = _unpack(w, dtype, n * m)
        return x @ (w.view(m, n) if col else w.view(n, m).t())

    if kind == "gemv":
        y = times(s["x"].double(), s["w"], case["n"], case["m"])
        y = y if s["bias"] is None else y + s["bias"].double()
        return y.cpu().numpy() if case["host"] else y
    if kind == "decode":
        x, kv = s["x"].double(), []
        h, d, f = case["hidden"], case["kv"], case["ffn"]
        for t in s["layers"]:
            a = _rms_norm(x, t["attn_norm"].double())
            kv.append((times(a, t["k"], d, h), times(a, t["v"], d, h)))
            o = times(times(a, t["q"], h, h), t["o"], h, h)
            b = _rms_norm(o, t["ffn_norm"].double())
            g = times(b, t["gate"], f, h)
            x = times(g * torch.sigmoid(g) * times(b, t["up"], f, h), t["down"], h, f)
        return {"y": x, "kv": kv}
    if kind == "mlp":
        h, f, col = case["hidden"], case["ffn"], case["col"]
        x = _rms_norm(s["x"].double(), s["norm"].double())
        g = times(x, s["gate"], f, h, col)
        return times(g * torch.sigmoid(g) * times(x, s["up"], f, h, col), s["down"], h, f, col)
    if kind == "head":
        x = s["x"].double()
        v, rows = case["vocab"], 16384
        out = []
        per = s["w"].numel() // v  # hidden is a whole number of blocks
        for r in range(0, v, rows):
            c = min(rows, v - r)
            out.append(times(x, s["w"][r * per:(r + c) * per], c, case["hidden"]))
        return torch.cat(out, dim=1)
    q = _pack(s["data"], dtype)
    return {"q": q, "back": _unpack(q, dtype, s["data"].numel() // 32 * 32)}
