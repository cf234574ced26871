"""The calls whose speed this framework is measured by, one dict each, with their inputs, the
work they cannot do without and the values they should return.

A case is one call (or one fixed sequence of calls) of the public API of ``mx_qlinear`` as a DiT
program makes it: a quantized linear layer, an FFN, or the norm + projection half of a block. The
token counts run from one (a timestep or modulation vector) over prompts (tens to hundreds) and
still images (thousands) to the 75600 tokens of 720p x 5 s; the layer shapes are those of the
workloads of ``bench.py``: hidden 5376 with attention 7168, QKV 21504 and a 14336 SwiGLU (ConvRot
256 on every layer), and hidden 5120 with QKV 15360 and a 20480 tanh-GELU FFN, plus 3072.
"""

from __future__ import annotations

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "x-minimaxh3_amd"))

import mx_qlinear as mx  # noqa: E402

_DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}

# (in features, out features) of the layers a drawn linear case takes.
_LAYERS = ((5376, 21504), (7168, 5376), (14336, 5376), (5376, 28672), (5120, 15360), (5120, 5120),
           (20480, 5120), (3072, 3072), (3072, 12288))


def _linear(m, k, n, **more):
    return {"kind": "linear", "m": m, "k": k, "n": n, "dtype": "bf16", "convrot": 256, "act": "none",
            "bias": True, **more}


def listed():
    return [
        # one token through the QKV projection: the smallest call, a stream of the weight
        {"name": "linear_m1", **_linear(1, 5376, 21504)},
        # a short prompt through a W4A8 layer as the reference's checkpoints store it
        {"name": "w4a8_ref_m20", "kind": "w4a8_ref", "m": 20, "k": 5376, "n": 21504, "group": 16, "srel": "e4m3",
         "bias": True},
        # a 77-token prompt through the attention output projection
        {"name": "linear_m77", **_linear(77, 7168, 5376)},
        # the MLP half of a block on a 333-token prompt
        {"name": "h3_mlp_m333", "kind": "h3_mlp", "m": 333, "segments": 1},
        # group-128 int4 weights, a low-resolution latent, the activations quantized in the call
        {"name": "w4a8_g128_m512", "kind": "w4a8_g128", "m": 512, "k": 5120, "n": 10240, "group": 128,
         "prepared": True, "dtype": "bf16", "bias": False},
        # a plain W8A8 layer of a small DiT (no rotation)
        {"name": "linear_m1024", **_linear(1024, 3072, 3072, convrot=0)},
        # float16 activations at a ragged token count
        {"name": "linear_f16_m2310", **_linear(2310, 5120, 5120, convrot=0, dtype="f16")},
        # norm, modulation and QKV projection of a still image with its prompt (ragged, three segments)
        {"name": "h3_qkv_m4097", "kind": "h3_qkv", "m": 4097, "segments": 3},
        # group-128 int4 weights at a square size, activations already quantized
        {"name": "w4a8_g128_m8192", "kind": "w4a8_g128", "m": 8192, "k": 5120, "n": 5120, "group": 128,
         "prepared": True, "dtype": "int8", "bias": False},
        # the down projection of a short clip in the checkpoint's W4A8 format
        {"name": "w4a8_ref_m14321", "kind": "w4a8_ref", "m": 14321, "k": 14336, "n": 5376, "group": 16, "srel": "e4m3",
         "bias": True},
        # LayerNorm modulation and QKV of two samples of a 480p clip
        {"name": "adaln_qkv_m32760", "kind": "adaln_qkv", "m": 32760, "samples": 2},
        # the FFN of 720p x 5 s, the headline workload
        {"name": "ffn_m75600", "kind": "ffn", "m": 75600},
    ]


def _tokens(rng, lo, hi):
    """A token count spread evenly over the logarithm of [lo, hi], about half of them odd."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("linear", "linear", "linear", "w4a8_ref", "w4a8_ref", "w4a8_g128", "h3_qkv", "h3_mlp",
                       "adaln_qkv", "ffn"))
    if kind == "linear":
        k, n = rng.choice(_LAYERS)
        dtype = rng.choice(("bf16", "bf16", "bf16", "f16", "f32"))
        act = rng.choice(("none", "none", "none", "gelu_tanh", "swiglu")) if dtype != "f32" else "none"
        return _linear(_tokens(rng, 1, 40000), k, n, dtype=dtype, act=act, convrot=rng.choice((256, 256, 0)),
                       bias=rng.random() < 0.7)
    if kind == "w4a8_ref":
        k, n = rng.choice(_LAYERS)
        return {"kind": kind, "m": _tokens(rng, 1, 40000), "k": k, "n": n, "group": rng.choice((16, 16, 32, 64)),
                "srel": rng.choice(("e4m3", "e4m3", "f32")), "bias": rng.random() < 0.7}
    if kind == "w4a8_g128":
        k, n = rng.choice(_LAYERS)
        return {"kind": kind, "m": _tokens(rng, 1, 16000), "k": k, "n": n, "group": 128, "prepared": rng.random() < 0.7,
                "dtype": rng.choice(("bf16", "int8")), "bias": rng.random() < 0.5}
    if kind in ("h3_qkv", "h3_mlp"):
        m = _tokens(rng, 16, 40000)
        return {"kind": kind, "m": m, "segments": rng.randint(1, 3)}
    if kind == "adaln_qkv":
        s = rng.randint(1, 3)
        return {"kind": kind, "m": s * _tokens(rng, 16, 20000), "samples": s}
    return {"kind": "ffn", "m": _tokens(rng, 1, 75600)}


# ---------------------------------------------------------------------------------------
# inputs (plain torch, from the seed alone)
# ---------------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _activations(g, m, k, dtype):
    """Transformer activations: unit normal with 0.5 % of the channels 20 times larger."""
    x = torch.randn(m, k, generator=g, device="cuda")
    idx = torch.randperm(k, generator=g, device="cuda")[: -(-k * 5 // 1000)]
    x[:, idx] *= 20.0
    return x.to(dtype)


def _weight(g, n, k):
    """An INT8 layer's weight: N(0, 0.02) rows quantized by their maximum."""
    w = torch.randn(n, k, generator=g, device="cuda") * 0.02
    s = w.abs().amax(dim=1, keepdim=True) / 127.0
    return torch.round(w / s).to(torch.int8), s.reshape(-1)


def _vec(g, shape, std, dtype=torch.bfloat16):
    return (torch.randn(shape, generator=g, device="cuda") * std).to(dtype)


# The reference's 16-level table, which its W4A8 checkpoints carry.
_TABLE = (-0.980602, -0.794529, -0.638165, -0.500986, -0.377321, -0.263187, -0.155210, -0.050720,
          0.052541, 0.156985, 0.265284, 0.379533, 0.502636, 0.638953, 0.794876, 0.980671)


def _w4_storage(g, n, k, group, srel):
    """W4A8 storage of an N(0, 0.02) weight: nearest-level codes, group and channel scales."""
    table = torch.tensor(_TABLE, device="cuda")
    edges = (table[1:] + table[:-1]) / 2
    w = (torch.randn(n, k, generator=g, device="cuda") * 0.02).view(n, k // group, group)
    s = w.abs().amax(dim=-1, keepdim=True).clamp_min(1e-8)
    codes = torch.bucketize(w / s, edges)
    s_ch = (table[codes] * s).abs().amax(dim=(1, 2)) / 127.0
    s_rel = s.squeeze(-1) / s_ch[:, None]
    c = codes.view(n, k).to(torch.uint8)
    packed = (c[:, 0::2] | (c[:, 1::2] << 4)).view(torch.int8)
    return packed, s_rel.to(torch.float8_e4m3fn) if srel == "e4m3" else s_rel, s_ch, table


def _segments(m, count):
    """`count` consecutive token ranges (prompt, references, target), each with its modulation row."""
    cuts = [0] + [m * (2 * i + 1) // (4 * count) for i in range(1, count)] + [m]
    return tuple((a, b, i) for i, (a, b) in enumerate(zip(cuts[:-1], cuts[1:])) if b > a)


def _inputs(case, seed):
    g, kind, m = _gen(seed), case["kind"], case["m"]
    if kind == "linear":
        dt = _DTYPES[case["dtype"]]
        out = torch.float16 if dt == torch.float16 else torch.bfloat16
        w, ws = _weight(g, case["n"], case["k"])
        return {"x": _activations(g, m, case["k"] * (2 if case["act"] == "swiglu" else 1), dt), "w": w, "ws": ws,
                "b": _vec(g, case["n"], 0.01, out) if case["bias"] else None, "out": out}
    if kind == "w4a8_ref":
        q, sr, sc, table = _w4_storage(g, case["n"], case["k"], case["group"], case["srel"])
        return {"x": _activations(g, m, case["k"], torch.bfloat16), "q": q, "sr": sr, "sc": sc, "table": table,
                "b": _vec(g, case["n"], 0.01) if case["bias"] else None}
    if kind == "w4a8_g128":
        n, k, group = case["n"], case["k"], case["group"]
        q = torch.randint(-128, 128, (n, k // 2), generator=g, device="cuda", dtype=torch.int8)
        gs = (torch.randn(k // group, n, generator=g, device="cuda").abs() * 0.01).to(torch.float16)
        st = {"q": q, "gs": gs, "xs": None, "b": _vec(g, n, 0.01) if case["bias"] else None}
        st["x"] = _activations(g, m, k, torch.bfloat16)
        if case["dtype"] == "int8":
            st["x"], st["xs"] = _quantize(st["x"])
            st["xs"] = st["xs"].float()
        return st
    if kind == "ffn":
        w1, s1 = _weight(g, 20480, 5120)
        w2, s2 = _weight(g, 5120, 20480)
        return {"x": _activations(g, m, 5120, torch.bfloat16), "w1": w1, "s1": s1, "b1": _vec(g, 20480, 0.01),
                "w2": w2, "s2": s2, "b2": _vec(g, 5120, 0.01)}
    if kind == "adaln_qkv":
        w, ws = _weight(g, 15360, 5120)
        s = case["samples"]
        return {"x": _activations(g, m, 5120, torch.bfloat16), "scale": _vec(g, (s, 5120), 0.2),
                "shift": _vec(g, (s, 5120), 0.2), "w": w, "ws": ws, "b": _vec(g, 15360, 0.01)}
    d, rows = 5376, case["segments"]
    st = {"x": _activations(g, m, d, torch.bfloat16), "norm": 1.0 + _vec(g, d, 0.1), "scale": _vec(g, (rows, d), 0.2),
          "shift": _vec(g, (rows, d), 0.2), "segments": _segments(m, rows)}
    if kind == "h3_qkv":
        st["w"], st["ws"] = _weight(g, 21504, d)
        st["b"] = _vec(g, 21504, 0.01)
        return st
    st["gate"] = _vec(g, (rows, d), 0.5)
    st["w1"], st["s1"] = _weight(g, 28672, d)
    st["b1"] = _vec(g, 28672, 0.01)
    st["w2"], st["s2"] = _weight(g, d, 14336)
    st["b2"] = _vec(g, d, 0.01)
    return st


# ---------------------------------------------------------------------------------------
# the calls
# ---------------------------------------------------------------------------------------

def prepare(case, seed):
    st = _inputs(case, seed)
    st["case"] = case
    if case["kind"] == "ffn":  # the buffers a program keeps between its layers
        st["ws"] = mx.FfnWorkspace(case["m"], 5120, 20480, st["x"].device)
    if case["kind"] == "h3_mlp":  # load-time weight order
        st["fc1"] = mx.prepare_swiglu_fc1(st.pop("w1"), st.pop("s1"), st.pop("b1"))
    if case["kind"] == "w4a8_g128" and case["prepared"]:
        st["q"] = mx.prepare_w4a8_grouped(st["q"])
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "linear":
        return mx.int8_linear(st["x"], st["w"], st["ws"], st["b"], out_dtype=st["out"], convrot=bool(case["convrot"]),
                              convrot_groupsize=case["convrot"] or 256,
                              input_act=None if case["act"] == "none" else case["act"])
    if kind == "w4a8_ref":
        return mx.w4a8_int8_linear(st["x"], st["q"], st["sr"], st["sc"], st["table"], None, st["b"],
                                   group_size=case["group"], convrot_groupsize=256)
    if kind == "w4a8_g128":
        return mx.w4a8_grouped_linear(st["x"], st["q"], st["gs"], case["group"], bias=st["b"], x_scale=st["xs"])
    if kind == "ffn":
        return mx.int8_ffn_gelu(st["x"], st["w1"], st["s1"], st["b1"], st["w2"], st["s2"], st["b2"], workspace=st["ws"])
    if kind == "adaln_qkv":
        q, s = mx.adaln_quantize_int8(st["x"], st["scale"], st["shift"])
        return mx.int8_linear_prequantized(q, s, st["w"], st["ws"], st["b"])
    norm = (st["norm"], 1e-6)
    if kind == "h3_qkv":
        q, s = mx.rms_adaln_quantize_int8(st["x"], norm, st["shift"], st["scale"], st["segments"])
        return mx.int8_linear_prequantized(q, s, st["w"], st["ws"], st["b"])
    residual = st["x"].clone()  # the call updates its residual in place
    return mx.h3_mlp_(residual, norm, st["shift"], st["scale"], st["gate"], st["segments"], st["fc1"], st["w2"],
                      st["s2"], st["b2"])


# ---------------------------------------------------------------------------------------
# the work of a pass
# ---------------------------------------------------------------------------------------

def work(case):
    kind, m = case["kind"], case["m"]
    if kind == "linear":
        k, n = case["k"], case["n"]
        e = 4 if case["dtype"] == "f32" else 2
        return {"bytes": m * k * e * (2 if case["act"] == "swiglu" else 1) + n * k + 4 * n + 2 * n * case["bias"]
                + 2 * m * n, "flops": 2 * m * n * k}
    if kind == "w4a8_ref":
        k, n = case["k"], case["n"]
        sb = 1 if case["srel"] == "e4m3" else 4
        return {"bytes": 2 * m * k + n * k // 2 + sb * n * k // case["group"] + 4 * n + 2 * n * case["bias"] + 2 * m * n,
                "flops": 2 * m * n * k}
    if kind == "w4a8_g128":
        k, n = case["k"], case["n"]
        return {"bytes": m * k * (1 if case["dtype"] == "int8" else 2) + n * k // 2 + 2 * n * k // case["group"]
                + 2 * n * case["bias"] + 2 * m * n, "flops": 2 * m * n * k}
    if kind == "ffn":
        return {"bytes": 4 * m * 5120 + 2 * 5120 * 20480 + 6 * (5120 + 20480), "flops": 4 * m * 5120 * 20480}
    if kind == "adaln_qkv":
        return {"bytes": 2 * m * (5120 + 15360) + 5120 * 15360 + 6 * 15360 + 4 * case["samples"] * 5120,
                "flops": 2 * m * 5120 * 15360}
    if kind == "h3_qkv":
        return {"bytes": 2 * m * (5376 + 21504) + 5376 * 21504 + 6 * 21504 + 4 * case["segments"] * 5376,
                "flops": 2 * m * 5376 * 21504}
    return {"bytes": 4 * m * 5376 + 3 * 5376 * 14336 + 6 * (28672 + 5376) + 6 * case["segments"] * 5376,
            "flops": 6 * m * 5376 * 14336}


def tolerance(case):
    """The int8 products are exact, so two correct implementations differ by the last rounding of
    the output (8 or 11 significant bits) and, behind a norm, by the int8 values that a last-bit
    difference of its statistics moves by one step."""
    if case["kind"] == "linear" and case["dtype"] == "f16":
        return {"rel": 1e-3}
    return {"rel": 7e-3}


# ---------------------------------------------------------------------------------------
# the values, in 64 bits
# ---------------------------------------------------------------------------------------

def _quantize(v):
    """The per-token int8 grid of rows in their dtype: (values, scales), the scale taken as
    max |v| / 127 in float32 and applied rounded to the rows' dtype."""
    s = (v.abs().amax(dim=-1, keepdim=True).double() / 127.0).float().clamp_min(1e-30)
    d = s.to(v.dtype)
    if v.dtype == torch.float16:
        d = torch.where(d == 0, torch.full_like(d, torch.finfo(torch.float16).tiny), d)
    q = torch.empty(v.shape, dtype=torch.int8, device=v.device)
    for a in range(0, v.shape[0], 8192):
        r = (v[a:a + 8192].double() / d[a:a + 8192].double()).to(v.dtype)
        q[a:a + 8192] = r.double().round().clamp(-128, 127).to(torch.int8)
    return q, s


def _rotate(v):
    """Each 256-column group times the regular Hadamard matrix, rounded once to the dtype."""
    h4 = torch.tensor([[1, 1, 1, -1], [1, 1, -1, 1], [1, -1, 1, 1], [-1, 1, 1, 1]], dtype=torch.float64, device=v.device)
    h16 = torch.kron(h4, h4)
    h = torch.kron(h16, h16) / 16.0
    out = torch.empty_like(v)
    for a in range(0, v.shape[0], 8192):
        part = v[a:a + 8192]
        out[a:a + 8192] = (part.double().reshape(-1, 256) @ h).reshape(part.shape).to(v.dtype)
    return out


def _product(q, s, w, ws, b):
    y = torch.empty(q.shape[0], w.shape[0], dtype=torch.float64, device=q.device)
    wt = w.double().t()
    for a in range(0, q.shape[0], 8192):
        y[a:a + 8192] = (q[a:a + 8192].double() @ wt) * s[a:a + 8192].double() * ws.double()
    return y if b is None else y.add_(b.double())


def _act(v, name):
    if name == "gelu_tanh":
        return torch.cat([torch.nn.functional.gelu(p.double(), approximate="tanh").to(v.dtype) for p in v.split(8192)])
    if name == "swiglu":
        parts = []
        for p in v.split(8192):
            gate, up = p.double().chunk(2, dim=-1)
            parts.append((torch.nn.functional.silu(gate).to(v.dtype).double() * up).to(v.dtype))
        return torch.cat(parts)
    return v


def _modulated(x, n, scale, shift, rows):
    parts = []
    for a in range(0, x.shape[0], 8192):
        r = rows[a:a + 8192]
        parts.append((n(x[a:a + 8192].double()) * (1.0 + scale.double())[r] + shift.double()[r]).to(x.dtype))
    return torch.cat(parts)


def _row_of(case, st):
    r = torch.zeros(case["m"], dtype=torch.int64, device="cuda")
    for a, b, row in st["segments"]:
        r[a:b] = row
    return r


def exact(case, seed):
    st, kind = _inputs(case, seed), case["kind"]
    if kind == "linear":
        v = _act(st["x"], case["act"])
        return _product(*_quantize(_rotate(v) if case["convrot"] else v), st["w"], st["ws"], st["b"])
    if kind == "w4a8_ref":
        n, k = case["n"], case["k"]
        u = st["q"].view(torch.uint8)
        codes = torch.stack([u & 15, u >> 4], dim=-1).reshape(n, k).long()
        grid = (st["table"][codes].view(n, -1, case["group"]) * st["sr"].float()[..., None]).double().round()
        return _product(*_quantize(_rotate(st["x"])), grid.clamp(-127, 127).view(n, k), st["sc"], st["b"])
    if kind == "w4a8_g128":
        n, k = case["n"], case["k"]
        u = st["q"].view(torch.uint8)
        codes = torch.stack([u & 15, u >> 4], dim=-1).reshape(n, -1, case["group"]).double() - 8.0
        w = (codes * st["gs"].double().t()[..., None]).view(n, k)
        q, s = (st["x"], st["xs"]) if case["dtype"] == "int8" else _quantize(st["x"])
        return _product(q, s, w, torch.ones(n, device="cuda"), st["b"])
    if kind == "ffn":
        h = _product(*_quantize(st["x"]), st["w1"], st["s1"], st["b1"]).to(torch.bfloat16)
        return _product(*_quantize(_act(h, "gelu_tanh")), st["w2"], st["s2"], st["b2"])
    if kind == "adaln_qkv":
        rows = torch.arange(case["m"], device="cuda") // (case["m"] // case["samples"])
        y = _modulated(st["x"], lambda v: torch.nn.functional.layer_norm(v, v.shape[-1:], eps=1e-6), st["scale"],
                       st["shift"], rows)
        return _product(*_quantize(y), st["w"], st["ws"], st["b"])
    rows = _row_of(case, st)
    w = st["norm"].double()
    y = _modulated(st["x"], lambda v: v * torch.rsqrt(v.square().mean(dim=-1, keepdim=True) + 1e-6) * w, st["scale"],
                   st["shift"], rows)
    q, s = _quantize(_rotate(y))
    if kind == "h3_qkv":
        return _product(q, s, st["w"], st["ws"], st["b"])
    h = _act(_product(q, s, st["w1"], st["s1"], st["b1"]).to(torch.bfloat16), "swiglu")
    y = _product(*_quantize(_rotate(h)), st["w2"], st["s2"], st["b2"])
    return st["x"].double() + y * st["gate"].double()[rows]
