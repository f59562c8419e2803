"""The calls that this library is measured on.

Each case is one operator call as an inference engine makes it: the operator,
the tensor descriptors and the workspace are made once per layer (`prepare`),
the call itself is repeated (`run`). The kinds are the layers of a quantized
transformer; the rows of A run from one token over decode batches and short
prompts to a long prefill, the widths are those of the 4096-wide model with
11008 / 14336-wide feed-forward layers that the repository's benchmark uses,
with other widths, odd ones among them, in the drawn cases.
"""
import math

import torch

import nnops_amd as na

DEV = "cuda"

WIDTHS = (1024, 4096, 11008, 14336)
MOST_FLOPS = 1.2e11


def listed():
    return [
        # the smallest call: one projection of a small model over a short
        # prompt, MatMul with its weight as [K, N], integer sums out
        dict(name="i8_matmul_small", kind="i8_matmul", m=128, k=1024, n=1024),
        # one token through a W8A8 layer whose output goes on in f16
        dict(name="i8_linear_decode", kind="i8_linear", m=1, k=4096, n=11008, out="f16"),
        # a decode batch of a serving engine through the down projection,
        # requantized for the next int8 layer
        dict(name="i8_linear_batch", kind="i8_linear", m=24, k=11008, n=4096, out="s8"),
        # a long prefill, requantized
        dict(name="i8_linear_prefill", kind="i8_linear", m=4096, k=4096, n=4096, out="s8"),
        # a ragged prompt through an int8 feed-forward layer, GELU before the
        # requantization, rows of padded buffers
        dict(name="i8_linear_gelu", kind="i8_gelu", m=333, k=4096, n=14336, pad=64),
        # one token through the down projection of a Q4_1 model
        dict(name="q4_linear_decode", kind="q4_linear", m=1, k=14336, n=4096, bias=False),
        # a small decode batch through the up projection
        dict(name="q4_linear_batch", kind="q4_linear", m=8, k=4096, n=14336, bias=False),
        # a short prompt through an attention projection with a bias
        dict(name="q4_linear_prompt", kind="q4_linear", m=77, k=4096, n=4096, bias=True),
        # a prefill chunk through the gated feed-forward layer (SwiGLU)
        dict(name="q4_gated_prefill", kind="q4_gated", m=512, k=4096, n=14336),
        # a layer that was left in f16, over a decode batch
        dict(name="fp_linear_batch", kind="fp_linear", m=40, k=4096, n=4096, bias=False),
        # f16 activations with calibrated per-token scales against an int8
        # weight (quantized on the way in, dequantized on the way out)
        dict(name="w8a8_matmul_prefill", kind="w8a8", m=1000, k=4096, n=11008),
        # activations to int8 and back between layers, a scale per token
        dict(name="qdq_roundtrip", kind="qdq", m=2048, k=4096),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, step):
    """Mostly a model's width, else any multiple of `step`."""
    if rng.random() < 0.6:
        return rng.choice(WIDTHS)
    return max(step, _log_int(rng, 512, 14336) // step * step)


def draw(rng):
    kind = rng.choice(("i8_matmul", "i8_linear", "i8_linear", "i8_gelu", "q4_linear", "q4_linear", "q4_gated",
                       "fp_linear", "w8a8", "qdq"))
    # K: whole Q4_1 blocks, 16-byte int8 or f16 rows; N: now and then odd
    c = dict(kind=kind, m=_log_int(rng, 1, 4096), k=_width(rng, 32))
    if kind != "qdq":
        c["n"] = _width(rng, rng.choice((1, 4, 64, 64)))
        flops = 2.0 * c["k"] * c["n"] * (2 if kind == "q4_gated" else 1)
        c["m"] = max(1, min(c["m"], int(MOST_FLOPS / flops)))
    if kind == "i8_linear":
        c["out"] = rng.choice(("s8", "f16", "s32"))
    if kind == "i8_gelu":
        c["pad"] = rng.choice((0, 64))
    if kind in ("q4_linear", "fp_linear"):
        c["bias"] = rng.random() < 0.25
    return c


# --- inputs ------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _normal(g, *shape):
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32)


def _rows_s8(x):
    """Symmetric int8 rows and their scales."""
    s = (x.abs().amax(dim=1) / 127.0).clamp_min(1e-8)
    return torch.round(x / s[:, None]).clamp_(-127, 127).to(torch.int8), s


def _q4_1(w):
    """Rows [n, k] to block_q4_1 bytes [n, k / 32 * 20] and the f16 d, m and
    whole q that they hold."""
    n, k = w.shape
    b = w.view(n, k // 32, 32)
    lo, hi = b.amin(dim=2), b.amax(dim=2)
    d = ((hi - lo) / 15.0).half()
    m = lo.half()
    q = torch.round((b - m.float()[..., None]) / d.float().clamp_min(1e-8)[..., None]).clamp_(0, 15).to(torch.uint8)
    out = torch.empty((n, k // 32, 20), dtype=torch.uint8, device=w.device)
    out[..., 0:2] = d[..., None].view(torch.uint8)
    out[..., 2:4] = m[..., None].view(torch.uint8)
    out[..., 4:20] = q[..., :16] | (q[..., 16:] << 4)
    return out.view(n, k // 32 * 20), d, m, q


def _padded(x, pad):
    if not pad:
        return x
    full = torch.zeros((x.shape[0], x.shape[1] + pad), dtype=x.dtype, device=x.device)
    full[:, :x.shape[1]] = x
    return full[:, :x.shape[1]]


def _inputs(case, seed):
    g = _gen(seed)
    kind, m, k = case["kind"], case["m"], case["k"]
    d = {}
    if kind == "qdq":
        x = _normal(g, m, k) * torch.exp(0.5 * _normal(g, m, 1))
        _, s = _rows_s8(x)
        d.update(x=x.half(), s=s, zp=torch.zeros(m, dtype=torch.int8, device=DEV))
        return d
    n = case["n"]
    rows = 2 * n if kind == "q4_gated" else n
    w = _normal(g, rows, k) * (1.0 / math.sqrt(k))
    x = _normal(g, m, k)
    if kind in ("i8_matmul", "i8_linear", "i8_gelu"):
        # calibrated per-tensor activation scale, per-channel weight scales;
        # a real product of these is about a standard normal
        s_a = 4.0 / 127.0
        d["x"] = torch.round(x / s_a).clamp_(-128, 127).to(torch.int8)
        d["w"], d["s_w"] = _rows_s8(w)
        d["s_a"] = s_a
        b = 0.1 * _normal(g, n)
        if case.get("out") == "f16":
            d["bias"] = b.half()
        else:
            d["bias"] = torch.round(b / (s_a * d["s_w"])).to(torch.int32)
        if kind == "i8_matmul":
            d["w"] = d["w"].t().contiguous()
    elif kind == "w8a8":
        _, d["s_x"] = _rows_s8(x)
        d["x"] = x.half()
        q, d["s_w"] = _rows_s8(w)
        d["w"] = q.t().contiguous()
    elif kind == "fp_linear":
        d["x"], d["w"] = x.half(), w.half()
    else:
        d["x"] = x.half()
        d["w"], d["d"], d["m"], d["q"] = _q4_1(w)
    if kind == "q4_gated" or (kind in ("q4_linear", "fp_linear") and case["bias"]):
        d["bias"] = (0.1 * _normal(g, rows)).half()
    return d


# s8 outputs cover about +-4 standard deviations of the product
S_OUT = 4.0 / 127.0


def prepare(case, seed):
    kind, m, k = case["kind"], case["m"], case["k"]
    d = _inputs(case, seed)
    if kind == "qdq":
        q = torch.empty((m, k), dtype=torch.int8, device=DEV)
        y = torch.empty((m, k), dtype=torch.float16, device=DEV)
        s, zp = na.tensor(d["s"]), na.tensor(d["zp"])
        qop, dop = na.QuantizeLinear(axis=0, output_dtype=na.DT_S8), na.DequantizeLinear(axis=0, output_dtype=na.DT_F16)
        return dict(calls=[(qop, [na.tensor(q)], [na.tensor(d["x"]), s, zp], None),
                           (dop, [na.tensor(y)], [na.tensor(q), s, zp], None)], out=[q, y])
    n = case["n"]
    if kind == "i8_matmul":
        y = torch.empty((m, n), dtype=torch.int32, device=DEV)
        op = na.MatMul(output_dtype=na.DT_S32)
        ins = [na.tensor(d["x"], scale=d["s_a"]), na.tensor(d["w"], scale_data=d["s_w"], granularity=2),
               na.tensor(d["bias"])]
        outs = [na.tensor(y)]
    elif kind in ("i8_linear", "i8_gelu"):
        out = case.get("out", "s8")
        tdt, dt = {"s8": (torch.int8, na.DT_S8), "s32": (torch.int32, na.DT_S32),
                   "f16": (torch.float16, na.DT_F16)}[out]
        pad = case.get("pad", 0)
        x = _padded(d["x"], pad)
        y = _padded(torch.empty((m, n), dtype=tdt, device=DEV), pad)
        if kind == "i8_gelu":
            op = na.Linear(output_dtype=dt, act=na.EP_GELU, float_epilogue=True)
        else:
            op = na.Linear(output_dtype=dt, act=na.EP_RELU if out == "s8" else None)
        ins = [na.tensor(x, scale=d["s_a"]), na.tensor(d["w"], scale_data=d["s_w"], granularity=2),
               na.tensor(d["bias"])]
        outs = [na.tensor(y, scale=S_OUT)]
    elif kind == "w8a8":
        y = torch.empty((m, n), dtype=torch.float16, device=DEV)
        op = na.MatMul(output_dtype=na.DT_F16)
        ins = [na.tensor(d["x"], scale_data=d["s_x"], granularity=1),
               na.tensor(d["w"], scale_data=d["s_w"], granularity=2)]
        outs = [na.tensor(y)]
        # the weight is laid out once, at load time
        _, packed = op.prepack(ins[1])
        ins[1] = packed
    else:
        y = torch.empty((m, n), dtype=torch.float16, device=DEV)
        if kind == "q4_gated":
            op = na.Linear(output_dtype=na.DT_F16, gated=True, gate_activation=na.EP_SILU)
        else:
            op = na.Linear(output_dtype=na.DT_F16)
        rows = 2 * n if kind == "q4_gated" else n
        ins = [na.tensor(d["x"]),
               na.tensor(d["w"], dtype=na.DT_Q4_1, shape=[rows, k]) if kind != "fp_linear" else na.tensor(d["w"])]
        if "bias" in d:
            ins.append(na.tensor(d["bias"]))
        outs = [na.tensor(y)]
    size = op.workspace_size(ins, outs)
    ws = torch.empty(size, dtype=torch.uint8, device=DEV) if size else None
    # (the library sizes the buffer; it needs no particular contents)
    return dict(calls=[(op, outs, ins, ws)], out=y, keep=d)


def run(state):
    for op, outs, ins, ws in state["calls"]:
        rc = op.compute(outs, ins, workspace=ws)
        if rc != na.OK:
            raise RuntimeError(f"compute failed: status {rc}")
    return state["out"]


# --- what a call cannot do without, and what it should give -------------------

def work(case):
    kind, m, k = case["kind"], case["m"], case["k"]
    if kind == "qdq":
        return {"bytes": m * k * (2 + 1 + 1 + 2) + 2 * m * 5, "flops": 0}
    n = case["n"]
    rows = 2 * n if kind == "q4_gated" else n
    a = {"i8_matmul": 1, "i8_linear": 1, "i8_gelu": 1}.get(kind, 2)
    w = {"q4_linear": 20 / 32, "q4_gated": 20 / 32, "fp_linear": 2}.get(kind, 1)
    o = {"i8_matmul": 4, "i8_gelu": 1}.get(kind) or {"s8": 1, "s32": 4, "f16": 2}[case.get("out", "f16")]
    tables = {"i8_matmul": 4 * n, "i8_linear": 8 * n, "i8_gelu": 8 * n, "w8a8": 4 * n + 4 * m,
              "q4_gated": 2 * rows}.get(kind, 2 * n if case.get("bias") else 0)
    return {"bytes": int(m * k * a + rows * k * w + m * n * o + tables), "flops": 2.0 * m * rows * k}


def tolerance(case):
    kind = case["kind"]
    if kind in ("i8_matmul", "i8_gelu", "qdq"):
        return "exact"          # integers; the dequantized values are one f32 product rounded to f16
    if kind == "i8_linear":
        # the f16 destination rounds one f32 value of an exact integer sum
        return "exact" if case["out"] != "f16" else {"rel": 2e-4}
    if kind == "w8a8":
        return {"rel": 2e-4}
    if kind == "fp_linear":
        return {"rel": 1e-3}    # f32 sums in any order, one rounding to f16
    # Q4_1: the decoded weight may be rounded to f16 (2^-12 of the weight and
    # its offset), f32 sums in any order, one rounding to f16
    return {"rel": 1.5e-3}


def exact(case, seed):
    kind, m, k = case["kind"], case["m"], case["k"]
    d = _inputs(case, seed)
    f64 = torch.float64
    if kind == "qdq":
        s = d["s"].to(f64)[:, None]
        q = torch.round(d["x"].to(f64) / s).clamp(-128, 127)
        return [q.to(torch.int8), q * s]
    if kind in ("i8_matmul", "i8_linear", "i8_gelu"):
        w = d["w"].to(f64)
        acc = d["x"].to(f64) @ (w if kind == "i8_matmul" else w.t().contiguous())
        s = d["s_w"].to(f64)[None, :] * d["s_a"]
        out = case.get("out", "s32" if kind == "i8_matmul" else "s8")
        if out == "f16":
            return acc * s + d["bias"].to(f64)
        acc = acc + d["bias"].to(f64)
        if out == "s32":
            return acc.to(torch.int32)
        f = acc * s
        if kind == "i8_gelu":
            f = 0.5 * f * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (f + 0.044715 * f * f * f)))
        else:
            f = f.clamp_min(0.0)
        f = f / S_OUT
        return (torch.sign(f) * torch.floor(f.abs() + 0.5)).clamp(-128, 127).to(torch.int8)
    if kind == "w8a8":
        s = d["s_x"].to(f64)[:, None]
        q = torch.round(d["x"].to(f64) / s).clamp(-128, 127)
        return (q @ d["w"].to(f64)) * s * d["s_w"].to(f64)[None, :]
    if kind == "fp_linear":
        y = d["x"].to(f64) @ d["w"].to(f64).t().contiguous()
        return y + d["bias"].to(f64) if "bias" in d else y
    w = (d["q"].to(f64) * d["d"].to(f64)[..., None] + d["m"].to(f64)[..., None]).view(-1, k)
    y = d["x"].to(f64) @ w.t().contiguous()
    if "bias" in d:
        y = y + d["bias"].to(f64)
    if kind == "q4_gated":
        gate, value = y[:, :case["n"]], y[:, case["n"]:]
        return gate * torch.sigmoid(gate) * value
    return y
