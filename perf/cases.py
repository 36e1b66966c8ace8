"""The workloads this library is timed on: the quantized matmuls of a decoder,
called as a program calls them, over the sizes, formats and options in use.

`listed()` holds the named cases, `draw(rng)` makes further ones of the same
families and ranges.  `prepare` builds what a program has in hand before the
call (packed weights, activations, output buffers), `run` makes one pass
through the public entry points of quixicore_hip, `exact` gives the same
outputs in 64-bit arithmetic from plain torch.

Families
  gemv       one decode projection (M = 1), f32 or per-block int8 activations
  layer      the projections of one decoder layer for one token, in the fused
             forms: Q/K/V with RoPE and cache insert, output projection,
             activation(gate) * up, down projection
  gemm       q8_0 / q4_0 weights against M activation rows: batched decode
             (M up to 32), short prompts, prefill
  canonical  canonical int8 weights with row or group scales and optional zero
             points, f32 / f16 / bf16 storage: a projection with bias and
             activation, or SwiGLU over gate and up
  w8a8_mlp   int8 x int8 prefill: residual add + RMS norm + quantization, up
             projection, per-token quantization, down projection
  w8a8_azp   int8 x int8 with asymmetric per-token activations
  load       packing f32 weights into blocks, and unpacking them again
"""
from __future__ import annotations

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "quixicore-cpu_amd"))
import quixicore_hip as qc  # noqa: E402

FORMAT = {"q8_0": qc.Q8_0, "q4_0": qc.Q4_0}
TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
ACTIVATION = {"none": 0, "gelu": 1, "gelu_tanh": 2, "silu": 3, "relu2": 4}
MAX_POSITION, SLOTS, EPS = 256, 64, 1e-5


# --------------------------------------------------------------------------
# Cases
# --------------------------------------------------------------------------
def listed():
    return [
        # the smallest call: one square projection of one token
        {"name": "gemv_q8_4096", "kind": "gemv", "format": "q8_0", "activations": "f32",
         "n": 4096, "k": 4096},
        # the longest rows, with activations quantized in the call
        {"name": "gemv_int8_q4_down", "kind": "gemv", "format": "q4_0", "activations": "int8",
         "n": 4096, "k": 14336},
        # single-stream decode: everything a layer multiplies for one token
        {"name": "decode_layer_q4", "kind": "layer", "format": "q4_0", "heads": 32, "kv_heads": 32,
         "head_dim": 128, "hidden": 4096, "ffn": 14336, "gelu": False},
        # batched decode of a few requests
        {"name": "batch8_q8_4096", "kind": "gemm", "format": "q8_0", "m": 8, "n": 4096, "k": 4096},
        # batched decode of many requests, the wide projection
        {"name": "batch32_q4_up", "kind": "gemm", "format": "q4_0", "m": 32, "n": 14336, "k": 4096},
        # a short prompt through a model of no round sizes
        {"name": "ragged_q8", "kind": "gemm", "format": "q8_0", "m": 77, "n": 5461, "k": 2752},
        # prefill of a prompt, and of a large batch of prompts
        {"name": "prefill512_q4_up", "kind": "gemm", "format": "q4_0", "m": 512, "n": 14336,
         "k": 4096},
        {"name": "prefill2048_q8_up", "kind": "gemm", "format": "q8_0", "m": 2048, "n": 14336,
         "k": 4096},
        # imported int8 checkpoint, batched decode: SwiGLU, affine groups, bf16 model
        {"name": "swiglu16_g128_bf16", "kind": "canonical", "swiglu": True, "m": 16, "n": 14336,
         "k": 4096, "group": 128, "zeros": True, "storage": "bf16", "activation": "none",
         "bias": False},
        # imported int8 checkpoint, prefill: row scales, bias and GELU, f16 model
        {"name": "gelu512_f16", "kind": "canonical", "swiglu": False, "m": 512, "n": 4096,
         "k": 4096, "group": 0, "zeros": False, "storage": "f16", "activation": "gelu",
         "bias": True},
        # the largest: an int8 MLP over 2048 tokens
        {"name": "w8a8_mlp_2048", "kind": "w8a8_mlp", "m": 2048, "hidden": 4096, "ffn": 14336},
        # asymmetric activations, a prompt of odd length
        {"name": "w8a8_azp_301", "kind": "w8a8_azp", "m": 301, "n": 4096, "k": 4096},
    ]


def _log(rng, low, high, step=1):
    """A size whose logarithm is uniform, rounded to a multiple of step."""
    v = math.exp(rng.uniform(math.log(low), math.log(high)))
    return max(step, int(round(v / step)) * step)


MOST_MNK = 2048 * 14336 * 4096


def draw(rng):
    kind = rng.choice(["gemv", "layer", "gemm", "gemm", "gemm", "canonical", "canonical",
                       "w8a8_mlp", "w8a8_azp", "load"])
    fmt = rng.choice(["q8_0", "q4_0"])
    if kind == "gemv":
        return {"kind": kind, "format": fmt, "activations": rng.choice(["f32", "f32", "int8"]),
                "n": _log(rng, 512, 32768), "k": _log(rng, 512, 16384, 32)}
    if kind == "layer":
        head_dim = rng.choice([64, 128])
        kv = rng.choice([2, 4, 8, 16])
        heads = kv * rng.choice([1, 2, 4])
        hidden = heads * head_dim
        return {"kind": kind, "format": fmt, "heads": heads, "kv_heads": kv, "head_dim": head_dim,
                "hidden": hidden, "ffn": _log(rng, 2 * hidden, 4 * hidden, 64),
                "gelu": rng.random() < 0.5}
    if kind == "gemm":
        k = _log(rng, 512, 14336, 64)
        n = _log(rng, 512, 16384)
        m = min(_log(rng, 2, 2048), MOST_MNK // (n * k))
        return {"kind": kind, "format": fmt, "m": m, "n": n, "k": k}
    if kind == "canonical":
        group = rng.choice([0, 0, 32, 64, 128])
        k = _log(rng, 512, 8192, 128 if group else 64)
        n = _log(rng, 512, 16384)
        swiglu = rng.random() < 0.5
        m = min(_log(rng, 1, 512), MOST_MNK // ((8 if swiglu else 4) * n * k))
        return {"kind": kind, "swiglu": swiglu, "m": m, "n": n, "k": k, "group": group,
                "zeros": rng.random() < 0.5, "storage": rng.choice(["f32", "f16", "bf16"]),
                "activation": "none" if swiglu else rng.choice(list(ACTIVATION)),
                "bias": not swiglu and rng.random() < 0.5}
    if kind == "w8a8_mlp":
        hidden = _log(rng, 512, 4096, 64)
        return {"kind": kind, "m": _log(rng, 16, 2048), "hidden": hidden,
                "ffn": _log(rng, 2 * hidden, 3.5 * hidden, 64)}
    if kind == "w8a8_azp":
        return {"kind": kind, "m": _log(rng, 16, 2048), "n": _log(rng, 512, 8192),
                "k": _log(rng, 512, 8192, 64)}
    return {"kind": kind, "format": fmt, "n": _log(rng, 512, 16384), "k": _log(rng, 512, 8192, 32)}


# --------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------
class _Gen:
    """Seeded tensors of one case on the GPU."""

    def __init__(self, seed):
        self.dev = torch.device("cuda:0")
        self.g = torch.Generator(device=self.dev)
        self.g.manual_seed(seed)

    def normal(self, *shape, sigma=1.0):
        return torch.randn(*shape, generator=self.g, device=self.dev) * sigma

    def hidden(self, *shape):
        """Hidden states: N(0, 1) with 0.1% of the entries 20 times larger."""
        x = self.normal(*shape)
        hit = torch.rand(*shape, generator=self.g, device=self.dev) < 0.001
        return torch.where(hit, x * 20.0, x)

    def weights(self, n, k):
        return self.normal(n, k, sigma=0.02)


def _encode(fmt, w):
    """GGUF blocks of f32 weights [n][k] (n * k/32 * {34, 18} bytes): per 32
    columns an f16 scale, then int8 codes (q8_0) or 4-bit codes, element i in
    the low and i + 16 in the high half of byte i (q4_0)."""
    n, k = w.shape
    b = w.reshape(-1, 32)
    if fmt == "q8_0":
        d = b.abs().amax(1, keepdim=True) / 127.0
        inv = torch.where(d == 0, 0.0, 1.0 / d)
        q = (b * inv).round().clamp(-128, 127).to(torch.int8).view(torch.uint8)
    else:
        top = b.gather(1, b.abs().argmax(1, keepdim=True))
        d = top / -8.0
        inv = torch.where(d == 0, 0.0, 1.0 / d)
        u = ((b * inv).round() + 8.0).clamp(0, 15).to(torch.uint8)
        q = u[:, :16] | (u[:, 16:] << 4)
    return torch.cat([d.half().view(torch.uint8), q], dim=1).reshape(-1).contiguous()


def _decode(fmt, packed, n, k):
    """The weights that _encode's blocks stand for, in 64 bits."""
    blocks = packed.reshape(n * (k // 32), -1)
    d = blocks[:, :2].contiguous().view(torch.float16).double()
    q = blocks[:, 2:].contiguous()
    if fmt == "q8_0":
        v = q.view(torch.int8).double()
    else:
        v = torch.cat([q & 15, q >> 4], dim=1).double() - 8.0
    return (d * v).reshape(n, k)


def _packed(case, g, n, k):
    return _encode(case["format"], g.weights(n, k))


def _row_int8(w):
    """Symmetric int8 codes and scales of each row."""
    s = w.abs().amax(1) / 127.0
    return (w / s[:, None]).round().clamp(-127, 127).to(torch.int8), s


def _out(*shape, dtype=torch.float32):
    return torch.zeros(*shape, dtype=dtype, device="cuda:0")


def prepare(case, seed):
    g = _Gen(seed)
    s = {"case": case}
    kind = case["kind"]
    if kind == "gemv":
        n, k = case["n"], case["k"]
        s.update(w=_packed(case, g, n, k), x=g.hidden(k), y=_out(n), status=_out(1, dtype=torch.int32))
    elif kind == "layer":
        h, hd = case["hidden"], case["head_dim"]
        nq, nkv, f = case["heads"] * hd, case["kv_heads"] * hd, case["ffn"]
        angle = torch.arange(MAX_POSITION, device=g.dev)[:, None] * (
            10000.0 ** (-torch.arange(hd // 2, device=g.dev) / (hd // 2)))[None, :]
        s.update(wq=_packed(case, g, nq, h), wk=_packed(case, g, nkv, h), wv=_packed(case, g, nkv, h),
                 wo=_packed(case, g, h, nq), wu=_packed(case, g, f, h), wg=_packed(case, g, f, h),
                 wd=_packed(case, g, h, f), x=g.hidden(h), attn=g.normal(nq), x2=g.hidden(h),
                 cos=angle.cos().float().contiguous(), sin=angle.sin().float().contiguous(),
                 position=seed % MAX_POSITION, slot=seed % SLOTS,
                 keys=g.normal(SLOTS, nkv), values=g.normal(SLOTS, nkv),
                 q=_out(nq), o=_out(h), act=_out(f), down=_out(h))
    elif kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        s.update(w=_packed(case, g, n, k), x=g.hidden(m, k), y=_out(m, n))
    elif kind == "canonical":
        m, n, k = case["m"], case["n"], case["k"]
        groups = k // case["group"] if case["group"] else 1
        for i in range(2 if case["swiglu"] else 1):
            w = g.weights(n, k).reshape(n, groups, -1)
            if case["zeros"]:
                low, high = w.amin(2, keepdim=True), w.amax(2, keepdim=True)
                scale = (high - low) / 255.0
                zero = (-128.0 - low / scale).round()
                codes = (w / scale + zero).round().clamp(-128, 127)
                s["zero%d" % i] = zero.reshape(n, groups).contiguous()
            else:
                scale = w.abs().amax(2, keepdim=True) / 127.0
                codes = (w / scale).round().clamp(-127, 127)
                s["zero%d" % i] = None
            s["code%d" % i] = codes.to(torch.int8).reshape(n, k).contiguous()
            s["scale%d" % i] = scale.reshape(n, groups).contiguous()
        s.update(x=g.hidden(m, k).to(TORCH[case["storage"]]),
                 bias=g.normal(n, sigma=0.1) if case["bias"] else None,
                 y=_out(m, n, dtype=TORCH[case["storage"]]))
        s["weights"] = [qc.cint8_weights(s["code%d" % i], s["scale%d" % i], s["zero%d" % i], n, k,
                                         groups) for i in range(2 if case["swiglu"] else 1)]
    elif kind == "w8a8_mlp":
        m, h, f = case["m"], case["hidden"], case["ffn"]
        s["up"], s["up_scale"] = _row_int8(g.weights(f, h))
        s["down"], s["down_scale"] = _row_int8(g.weights(h, f))
        s.update(x=g.normal(m, h), residual=g.hidden(m, h), norm=1.0 + g.normal(h, sigma=0.1),
                 status=_out(1, dtype=torch.int32))
    elif kind == "w8a8_azp":
        s["w"], s["w_scale"] = _row_int8(g.weights(case["n"], case["k"]))
        s.update(row_sum=s["w"].sum(1, dtype=torch.int32), x=g.hidden(case["m"], case["k"]) + 0.25,
                 status=_out(1, dtype=torch.int32))
    else:
        n, k = case["n"], case["k"]
        size = qc.packed_size(FORMAT[case["format"]], n, k)[1]
        s.update(w=g.weights(n, k), packed=_out(size, dtype=torch.uint8), back=_out(n, k),
                 status=_out(1, dtype=torch.int32))
    return s


# --------------------------------------------------------------------------
# One pass
# --------------------------------------------------------------------------
def _ok(status):
    if status != 0:
        raise RuntimeError(f"status {status}: {qc.lib.qc_hip_last_error().decode()}")


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "gemv":
        fmt = FORMAT[case["format"]]
        if case["activations"] == "int8":
            _ok(qc.qgemv_w8a8_raw(fmt, s["w"], s["x"], s["y"], case["n"], case["k"], s["status"]))
        else:
            qc.qgemv(fmt, s["w"], s["x"], case["n"], case["k"], y=s["y"])
        return s["y"]
    if kind == "layer":
        fmt, h, f, hd = FORMAT[case["format"]], case["hidden"], case["ffn"], case["head_dim"]
        _ok(qc.qgemv_qkv_rope_kv_raw(fmt, s["wq"], s["wk"], s["wv"], s["x"], s["cos"], s["sin"],
                                     s["q"], s["keys"], s["values"], case["heads"],
                                     case["kv_heads"], hd, h, SLOTS, MAX_POSITION, s["position"],
                                     s["slot"]))
        qc.qgemv(fmt, s["wo"], s["attn"], h, case["heads"] * hd, y=s["o"])
        _ok(qc.qgemv_up_gate_activation_raw(fmt, s["wu"], s["wg"], s["x2"], s["act"], f, h,
                                            gelu_tanh=case["gelu"]))
        qc.qgemv(fmt, s["wd"], s["act"], h, f, y=s["down"])
        return [s["q"], s["keys"], s["values"], s["o"], s["act"], s["down"]]
    if kind == "gemm":
        return qc.qgemm(FORMAT[case["format"]], s["w"], s["x"], case["n"], case["k"], y=s["y"])
    if kind == "canonical":
        st = qc.STORAGE[case["storage"]]
        _ok(qc.cint8_project_raw(1 if case["swiglu"] else 0, s["weights"], s["x"], st, case["m"],
                                 [s["y"]], [st], bias=s["bias"],
                                 activation=ACTIVATION[case["activation"]]))
        return s["y"]
    if kind == "w8a8_mlp":
        codes, residual, scales = qc.rms_norm_add_quant_int8(s["x"], s["residual"], s["norm"], EPS,
                                                             dev_status=s["status"])
        up = qc.int8_gemm(s["up"], codes, s["up_scale"], scales.view(-1), dev_status=s["status"])
        codes2, scales2 = qc.quantize_int8(up, dev_status=s["status"])
        down = qc.int8_gemm(s["down"], codes2, s["down_scale"], scales2.view(-1),
                            dev_status=s["status"])
        return [codes, residual, scales, up, codes2, scales2, down]
    if kind == "w8a8_azp":
        codes, scales, zeros = qc.quantize_int8_asymmetric(s["x"], dev_status=s["status"])
        y = qc.int8_gemm(s["w"], codes, s["w_scale"], scales, row_sum=s["row_sum"], zp=zeros,
                         asymmetric=True, dev_status=s["status"])
        return [codes, scales, zeros, y]
    fmt, n, k = FORMAT[case["format"]], case["n"], case["k"]
    _ok(qc.pack_raw(fmt, s["w"], s["packed"], n, k, dev_status=s["status"]))
    _ok(qc.unpack_raw(fmt, s["packed"], s["back"], n, k))
    return [s["packed"], s["back"]]


# --------------------------------------------------------------------------
# What a pass cannot do without, and what its outputs may be off by
# --------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    bits = {"q8_0": 34 / 32, "q4_0": 18 / 32}.get(case.get("format"), 1.0)
    if kind == "gemv":
        n, k = case["n"], case["k"]
        return {"bytes": n * k * bits + 4 * (n + k), "flops": 2 * n * k}
    if kind == "layer":
        h, f = case["hidden"], case["ffn"]
        nq, nkv = case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"]
        weights = (2 * nq + 2 * nkv + 3 * f) * h
        return {"bytes": weights * bits + 4 * (4 * h + 2 * nq + 2 * nkv + 2 * f),
                "flops": 2 * weights}
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": n * k * bits + 4 * m * (n + k), "flops": 2 * m * n * k}
    if kind == "canonical":
        m, n, k, two = case["m"], case["n"], case["k"], 2 if case["swiglu"] else 1
        groups = k // case["group"] if case["group"] else 1
        side = n * groups * (8 if case["zeros"] else 4)
        size = 4 if case["storage"] == "f32" else 2
        return {"bytes": two * (n * k + side) + size * m * (n + k), "flops": 2 * two * m * n * k}
    if kind == "w8a8_mlp":
        m, h, f = case["m"], case["hidden"], case["ffn"]
        # x, residual in; residual, codes out and in; weights; up out and in;
        # its codes out and in; down out
        return {"bytes": 2 * h * f + m * (4 * 3 * h + 2 * h + 8 * f + 2 * f + 4 * h),
                "flops": 4 * m * h * f}
    if kind == "w8a8_azp":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": n * k + 4 * m * (n + k) + 2 * m * k, "flops": 2 * m * n * k}
    n, k = case["n"], case["k"]
    return {"bytes": n * k * (8 + 2 * bits), "flops": 0}


def tolerance(case):
    kind = case["kind"]
    if kind in ("w8a8_mlp", "w8a8_azp", "load"):
        return "exact"                    # defined bit for bit
    if kind == "gemv" and case["activations"] == "int8":
        return "exact"                    # integer block dots, summed in block order
    if kind == "canonical" and case["storage"] != "f32":
        # one rounding to the 16-bit output, of either side
        return {"rel": 4e-3, "max": 1e-2} if case["storage"] == "bf16" else {"rel": 5e-4, "max": 1.5e-3}
    return {"rel": 1e-5}                  # 22-bit (or two 8-bit) activations, 32-bit sums


# --------------------------------------------------------------------------
# The same outputs in 64 bits
# --------------------------------------------------------------------------
def _silu(v):
    return v / (1.0 + torch.exp(-v))


def _gelu_tanh(v):
    return 0.5 * v * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (v + 0.044715 * v ** 3)))


def _activate(name, v):
    if name == "gelu":
        return 0.5 * v * (1.0 + torch.erf(v / math.sqrt(2.0)))
    if name == "gelu_tanh":
        return _gelu_tanh(v)
    if name == "silu":
        return _silu(v)
    if name == "relu2":
        return v.clamp_min(0.0) ** 2
    return v


def _mv(case, w, x, n):
    return _decode(case["format"], w, n, x.numel()) @ x.double()


def _quantize_rows(x):
    """The codes and scales quantize_int8 is defined by: f32 arithmetic."""
    s = x.abs().amax(1) / 127.0
    q = torch.where(s[:, None] == 0, 0.0, x / s[:, None]).round().clamp(-127, 127)
    return q, s


def _int8_product(x, w, x_scale, w_scale):
    acc = x.double() @ w.double().T.contiguous()
    return acc * w_scale.double()[None, :] * x_scale.double()[:, None]


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "gemv":
        n, k = case["n"], case["k"]
        if case["activations"] == "f32":
            return _mv(case, s["w"], s["x"], n)
        q, d = _quantize_rows(s["x"].reshape(-1, 32))
        x = (q.double() * d.double()[:, None]).reshape(-1)
        return _decode(case["format"], s["w"], n, k) @ x
    if kind == "layer":
        h, f, hd = case["hidden"], case["ffn"], case["head_dim"]
        nq, nkv = case["heads"] * hd, case["kv_heads"] * hd
        c, sn = s["cos"][s["position"]].double(), s["sin"][s["position"]].double()

        def rotate(v):
            a, b = v.reshape(-1, 2, hd // 2).unbind(1)
            return torch.stack([a * c - b * sn, b * c + a * sn], dim=1).reshape(-1)

        keys, values = s["keys"].double(), s["values"].double()
        q = rotate(_mv(case, s["wq"], s["x"], nq))
        keys[s["slot"]] = rotate(_mv(case, s["wk"], s["x"], nkv))
        values[s["slot"]] = _mv(case, s["wv"], s["x"], nkv)
        up, gate = _mv(case, s["wu"], s["x2"], f), _mv(case, s["wg"], s["x2"], f)
        act = (_gelu_tanh(gate) if case["gelu"] else _silu(gate)) * up
        return [q, keys, values, _mv(case, s["wo"], s["attn"], h), act,
                _mv(case, s["wd"], act, h)]
    if kind == "gemm":
        return s["x"].double() @ _decode(case["format"], s["w"], case["n"], case["k"]).T.contiguous()
    if kind == "canonical":
        n, k = case["n"], case["k"]
        ys = []
        for i in range(2 if case["swiglu"] else 1):
            scale = s["scale%d" % i].double()[:, :, None]
            code = s["code%d" % i].double().reshape(n, scale.shape[1], -1)
            if case["zeros"]:
                code = code - s["zero%d" % i].double()[:, :, None]
            ys.append(s["x"].double() @ (code * scale).reshape(n, k).T.contiguous())
        if case["swiglu"]:
            return _silu(ys[0]) * ys[1]
        return _activate(case["activation"], ys[0] + (s["bias"].double() if case["bias"] else 0.0))
    if kind == "w8a8_mlp":
        # codes follow from f32 steps in a stated order, so only what is
        # defined by the inputs alone has a 64-bit value
        return [None, s["x"].double() + s["residual"].double(), None, None, None, None, None]
    if kind == "w8a8_azp":
        x = s["x"].double()
        low, high = x.amin(1), x.amax(1)
        scale = ((high - low) / 255.0).float().double()
        zero = (-128.0 - low / scale).round()
        q = ((x / scale[:, None]).round() + zero[:, None]).clamp(-128, 127)
        y = (q - zero[:, None]) @ s["w"].double().T.contiguous()
        return [None, scale, None, y * s["w_scale"].double()[None, :] * scale[:, None]]
    blocks = _encode(case["format"], s["w"])
    return [None, _decode(case["format"], blocks, case["n"], case["k"])]
