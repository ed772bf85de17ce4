"""Performance cases of the quantized-linear framework: what a user's program has it do.

Three kinds of work: the quantized linears of a diffusion transformer (one call per layer and step:
rotate, per-token quantize, integer GEMM, scales and bias), the standalone rotate + quantize kernel, and
the two directions of weight storage (quantizing a float weight for a checkpoint, decoding a shipped
checkpoint's weight at load). Sizes are the benchmark's configurations (hidden 3072, MLP ratio 4 or FFN
14336, adaLN modulation at one row, 256 or 77 text tokens, 1024 / 4096 / 4352 / 32760 image or video
tokens) and ragged ones between them.

Weights are generated in the stored, quantized form, as a checkpoint holds them: Gaussian weights (a
rotated Gaussian weight is Gaussian again) quantized by the format's rule in plain torch. Activations are
N(0, 1) with 1 % of the channels x20 and, for the 4-bit activations, 0.1 % of the tokens x50.
"""
from __future__ import annotations

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "comfy-quant-bench_amd"))

import kitchen_amd as ck  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
GROUP = 64

# Linear formats: activations' bits, weights' bytes per element (codes with their scales and zero-points)
FORMATS = {
    "w4a8": (8, 0.5 + 2 / 64 + 0.5 / 64),   # uint4 asymmetric, fp16 scale and uint4 zero-point per 64
    "w4a4": (4, 0.5 + 2 / 64),              # int4 symmetric, fp16 scale per 64
    "w4a4row": (4, 0.5),                    # shipped ConvRot W4A4: int4, fp32 scale per row
    "w8a8": (8, 1.0),                       # int8, fp32 scale per row
}


def _linear(name, fmt, m, k, n, h=256, dtype="bf16", bias=True, act="none"):
    case = {"op": "linear", "fmt": fmt, "m": m, "k": k, "n": n, "h": h, "dtype": dtype, "bias": bias, "act": act}
    return dict(case, name=name) if name else case


def listed():
    return [
        # the adaLN modulation of one block: one conditioning vector, the smallest call of a step
        _linear("adaln_w4a8_m1", "w4a8", 1, 3072, 18432),
        # a short text prompt's attention projection: few rows, latency and weight reads
        _linear("prompt_w4a4_m77", "w4a4", 77, 3072, 3072, h=64),
        # the text stream of a joint block, MLP up
        _linear("text_w8a8_m256", "w8a8", 256, 3072, 12288),
        # a 512 x 512 image's attention projection
        _linear("attn_w4a8_m1024", "w4a8", 1024, 3072, 3072),
        # an odd aspect ratio's token count, fused QKV, fp16 model without bias
        _linear("qkv_w4a4_m2745", "w4a4", 2745, 3072, 9216, dtype="fp16", bias=False),
        # image + text tokens of a 1024 x 1024 image, MLP up
        _linear("mlp_up_w4a8_m4352", "w4a8", 4352, 3072, 12288),
        # image tokens, MLP down
        _linear("mlp_down_w8a8_m4096", "w8a8", 4096, 12288, 3072),
        # MLP down of a gated MLP in the shipped 4-bit format, the SwiGLU folded into its quantizer
        _linear("mlp_down_swiglu_w4a4row_m4096", "w4a4row", 4096, 12288, 3072, act="swiglu"),
        # the activation quantizer alone at a video's token count
        {"name": "rotquant_m32760", "op": "rotquant", "m": 32760, "k": 3072, "h": 256, "bits": 8, "dtype": "bf16",
         "act": "none"},
        # MLP down of a video model (the largest call)
        _linear("video_mlp_down_w4a8_m32760", "w4a8", 32760, 14336, 3072),
        # a converter quantizing one MLP weight for a checkpoint
        {"name": "convert_w4a8_12288", "op": "encode", "fmt": "w4a8", "k": 3072, "n": 12288, "h": 256, "dtype": "bf16"},
        # a loader decoding one shipped codebook weight
        {"name": "load_codebook_12288", "op": "decode", "k": 3072, "n": 12288, "gs": 16},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["linear"] * 7 + ["rotquant", "encode", "decode"])
    if op == "linear":
        fmt = rng.choice(["w4a8", "w4a4", "w8a8", "w4a4row"])
        h = rng.choice([16, 64, 256]) if fmt == "w4a4" else 256
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
        act = rng.choice(["none", "none", "none", "swiglu"]) if fmt in ("w4a4row", "w8a8") else "none"
        while True:
            m = rng.choice([1, _log_int(rng, 2, 128), _log_int(rng, 129, 32760), _log_int(rng, 129, 32760)])
            k, n = max(h, 64) * _log_int(rng, -(-1024 // max(h, 64)), 14336 // max(h, 64)), _log_int(rng, 1024, 18432)
            n = rng.choice([n, 64 * (n // 64)])
            if m * k * n <= 32760 * 14336 * 3072:
                return _linear(None, fmt, m, k, n, h, dtype, rng.random() < 0.7, act)
    if op == "rotquant":
        act = rng.choice(["none", "swiglu"])
        while True:
            m, k = _log_int(rng, 64, 32760), 256 * rng.randint(4, 56)
            if m * k <= 32760 * 3072:
                return {"op": op, "m": m, "k": k, "h": 256, "bits": rng.choice([4, 8]) if act == "none" else 4,
                        "dtype": rng.choice(["bf16", "fp16"]), "act": act}
    k, n = 256 * rng.randint(4, 48), _log_int(rng, 1024, 12288)
    if op == "encode":
        return {"op": op, "fmt": rng.choice(list(FORMATS)), "k": k, "n": n, "h": 256,
                "dtype": rng.choice(["bf16", "bf16", "fp32"])}
    return {"op": op, "k": k, "n": n, "gs": rng.choice([16, 32, 64])}


# ------------------------------------------------------------------------------------------- inputs

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _activations(m, k, dtype, spikes, gen):
    x = torch.randn(m, k, generator=gen, device=gen.device)
    x[:, torch.randperm(k, generator=gen, device=gen.device)[:max(1, k // 100)]] *= 20.0
    if spikes and m >= 16:
        x[torch.randperm(m, generator=gen, device=gen.device)[:max(1, m // 1000)]] *= 50.0
    return x.to(dtype)


def _pack(q):
    """4-bit codes [N, K], two per byte, the even column in the low nibble."""
    q = q.to(torch.int16) & 0xF
    return (q[:, 0::2] | (q[:, 1::2] << 4)).to(torch.uint8)


def _weight(fmt, n, k, gen):
    """A stored weight: the tensors a checkpoint holds, and its codes less their zero-points and scales
    for the 64-bit result."""
    w = torch.randn(n, k, generator=gen, device=gen.device) * 0.02
    if fmt == "w4a8":
        g = w.view(n, k // GROUP, GROUP)
        lo, hi = g.amin(2).clamp(max=0), g.amax(2).clamp(min=0)
        s = ((hi - lo) / 15).half()
        z = (-lo / s.float()).round().clamp(0, 15)
        q = ((g / s.float()[..., None]).round() + z[..., None]).clamp(0, 15)
        zp = z if z.shape[1] % 2 == 0 else torch.cat([z, z.new_zeros(n, 1)], 1)
        return {"q": _pack(q.view(n, k)), "s": s, "z": _pack(zp), "codes": (q - z[..., None]).view(n, k)}
    if fmt == "w4a4":
        g = w.view(n, k // GROUP, GROUP)
        s = (g.abs().amax(2) / 7).half()
        q = (g / s.float()[..., None]).round().clamp(-7, 7).view(n, k)
        return {"q": _pack(q).view(torch.int8), "s": s, "codes": q}
    top = 7 if fmt == "w4a4row" else 127
    s = w.abs().amax(1, keepdim=True).clamp(min=1e-10) / top
    q = (w / s).round().clamp(-top, top)
    if fmt == "w4a4row":
        return {"q": _pack(q).view(torch.int8), "s": s[:, 0].contiguous(), "codes": q}
    return {"q": q.to(torch.int8), "s": s, "codes": q}


def _inputs(case, seed):
    gen = torch.Generator(device=_device()).manual_seed(seed)
    k = case["k"]
    if case["op"] in ("linear", "rotquant"):
        spikes = case.get("bits", FORMATS.get(case.get("fmt"), (8,))[0]) == 4
        width = 2 * k if case["act"] == "swiglu" else k
        x = _activations(case["m"], width, DTYPES[case["dtype"]], spikes, gen)
        if case["op"] == "rotquant":
            return {"x": x}
        bias = (torch.randn(case["n"], generator=gen, device=gen.device) * 0.1).to(x.dtype) if case["bias"] else None
        return {"x": x, "bias": bias, **_weight(case["fmt"], case["n"], k, gen)}
    if case["op"] == "encode":
        return {"w": (torch.randn(case["n"], k, generator=gen, device=gen.device) * 0.02).to(DTYPES[case["dtype"]])}
    # a shipped codebook weight: 16 levels, fp8 group scales, fp32 row scales
    n, gs = case["n"], case["gs"]
    q = torch.randint(-128, 128, (n, k // 2), generator=gen, device=gen.device, dtype=torch.int8)
    s_rel = (torch.rand(n, k // gs, generator=gen, device=gen.device) * 40 + 10).to(torch.float8_e4m3fn)
    s_channel = torch.rand(n, generator=gen, device=gen.device) * 2e-4 + 3e-4
    codebook = torch.sort(torch.randn(16, generator=gen, device=gen.device).clamp(-2.5, 2.5))[0]
    return {"qdata": q, "s_rel": s_rel, "s_channel": s_channel, "codebook": codebook}


def prepare(case, seed):
    state = _inputs(case, seed)
    state.pop("codes", None)
    if case["op"] == "linear" and case["fmt"] == "w8a8" and case["k"] >= 192:
        state["q"] = ck.tile_int8_weight(state["q"])   # the loader holds int8 weights in the GEMM's tiles
    state["case"] = case
    return state


# ---------------------------------------------------------------------------------------------- run

def run(state):
    case = state["case"]
    if case["op"] == "linear":
        act = None if case["act"] == "none" else case["act"]
        if case["fmt"] == "w4a8":
            return ck.w4a8_int8_linear(state["x"], state["q"], state["s"], None, None, state["z"], state["bias"], GROUP,
                                       case["h"], DTYPES[case["dtype"]])
        if case["fmt"] == "w8a8":
            return ck.int8_linear(state["x"], state["q"], state["s"], state["bias"], DTYPES[case["dtype"]], True,
                                  case["h"], act)
        return ck.convrot_w4a4_linear(state["x"], state["q"], state["s"], state["bias"], case["h"], GROUP, "int4", act)
    if case["op"] == "rotquant":
        if case["act"] == "swiglu":
            return ck.swiglu_quantize_int4_rowwise_convrot64(state["x"], case["h"])
        if case["bits"] == 4:
            return ck.quantize_int4_rowwise_convrot64(state["x"], case["h"])
        return ck.quantize_int8_rowwise_convrot(state["x"], case["h"])
    if case["op"] == "encode":
        w, fmt, h = state["w"], case["fmt"], case["h"]
        if fmt == "w4a8":
            return ck.quantize_w4a8_asym_weight(w, GROUP, h)
        if fmt == "w4a4":
            return ck.quantize_w4a4_group_weight(w, GROUP, h)
        if fmt == "w4a4row":
            return ck.quantize_convrot_w4a4_weight(w, h, GROUP)
        return ck.quantize_int8_convrot_weight(w, h)
    p = ck.PreparedW4A8(state["qdata"], state["s_rel"], state["s_channel"], state["codebook"], case["gs"])
    return p.q8, p.row_scale


def work(case):
    k = case["k"]
    if case["op"] == "linear":
        m, n = case["m"], case["n"]
        size = DTYPES[case["dtype"]].itemsize
        x = m * k * size * (2 if case["act"] == "swiglu" else 1)
        return {"bytes": x + n * k * FORMATS[case["fmt"]][1] + n * (4 + size) + m * n * size, "flops": 2.0 * m * n * k}
    if case["op"] == "rotquant":
        m = case["m"]
        return {"bytes": m * k * ((4 if case["act"] == "swiglu" else 2) + case["bits"] / 8) + 4 * m, "flops": 0.0}
    n = case["n"]
    if case["op"] == "encode":
        return {"bytes": n * k * (DTYPES[case["dtype"]].itemsize + FORMATS[case["fmt"]][1]) + 4 * n, "flops": 0.0}
    return {"bytes": n * k * (0.5 + 1 / case["gs"] + 1) + 8 * n, "flops": 0.0}


def tolerance(case):
    """Codes, scales and decoded weights are whole numbers or single IEEE operations: the same bytes. A
    linear's output differs from the 64-bit result by its rounding to the output type (2^-9 in bf16, 2^-12
    in fp16) and by the fp32 sums of the group scales (up to 4e-4 of the output's norm)."""
    if case["op"] != "linear":
        return "exact"
    grouped = case["fmt"] in ("w4a8", "w4a4")
    return {"rel": {"bf16": 6e-3, "fp16": 1.6e-3 if grouped else 8e-4, "fp32": 1.6e-3 if grouped else 2e-4}[case["dtype"]]}


# ------------------------------------------------------------------------------- 64-bit results

def _hadamard(block):
    """The orthonormal H_block: Kronecker powers of H_4 / 2, y_i = sum / 2 - x_{3 - i}."""
    h4 = 0.5 * torch.ones(4, 4, dtype=torch.float64) - torch.flip(torch.eye(4, dtype=torch.float64), (1,))
    h = h4
    while h.shape[0] < block:
        h = torch.kron(h4, h)
    return h


def _rotate(x, block):
    return (x.double().view(-1, block) @ _hadamard(block).to(x.device)).view(x.shape)


def _quantized(x, case, bits):
    """(codes, scales) of the activation rows in 64 bits."""
    if case["act"] == "swiglu":
        gate, up = x.double().chunk(2, dim=-1)
        x = (torch.nn.functional.silu(gate) * up).to(x.dtype)
    r = _rotate(x, case["h"])
    s = (r.abs().amax(1, keepdim=True) / (2 ** (bits - 1) - 1)).clamp(min=1e-10)
    return (r / s).round(), s


def exact(case, seed):
    t = _inputs(case, seed)
    if case["op"] == "linear":
        n, k = case["n"], case["k"]
        s = t["s"].double()
        w = (t["codes"].double().view(n, -1, GROUP) * s[..., None]).view(n, k) if s.dim() == 2 and s.shape[1] > 1 \
            else t["codes"].double() * s.view(n, 1)
        y = torch.empty(case["m"], n, dtype=torch.float64, device=w.device)
        for i in range(0, case["m"], 4096):
            q, sa = _quantized(t["x"][i:i + 4096], case, FORMATS[case["fmt"]][0])
            y[i:i + 4096] = (q @ w.T) * sa
        return y if t["bias"] is None else y.add_(t["bias"].double())
    if case["op"] == "rotquant":
        q, s = _quantized(t["x"], case, case["bits"])
        q = q.to(torch.int8)
        return (_pack(q).view(torch.int8) if case["bits"] == 4 else q), s[:, 0]
    if case["op"] == "encode":
        return _exact_encode(case, t["w"])
    q = t["qdata"].to(torch.int16) & 0xFF
    codes = torch.stack([q & 0xF, q >> 4], dim=2).view(case["n"], case["k"]).long()
    level = t["codebook"].double()[codes].view(case["n"], -1, case["gs"]) * t["s_rel"].double()[..., None]
    q8 = level.round().clamp(-127, 127).to(torch.int8).view(case["n"], case["k"])
    pad = -case["n"] % 16   # 16-row tiles of 64 columns, rows past N zero
    q8 = torch.cat([q8, q8.new_zeros(pad, case["k"])]) if pad else q8
    return q8.view(-1, 16, case["k"] // 64, 64).transpose(1, 2).contiguous(), t["s_channel"]


def _exact_encode(case, w):
    n, k, fmt = case["n"], case["k"], case["fmt"]
    r = _rotate(w, case["h"])
    if fmt == "w4a8":
        g = r.view(n, k // GROUP, GROUP)
        lo, hi = g.amin(2).clamp(max=0), g.amax(2).clamp(min=0)
        s = ((hi - lo) / 15).half()
        z = (-lo / s.double()).round().clamp(0, 15)
        q = ((g / s.double()[..., None]).round() + z[..., None]).clamp(0, 15).view(n, k)
        z = z if z.shape[1] % 2 == 0 else torch.cat([z, z.new_zeros(n, 1)], 1)
        return _pack(q), s, _pack(z)
    if fmt == "w4a4":
        g = r.view(n, k // GROUP, GROUP)
        s = (g.abs().amax(2) / 7).half()
        return _pack((g / s.double()[..., None]).round().clamp(-7, 7).view(n, k)).view(torch.int8), s
    top = 7 if fmt == "w4a4row" else 127
    s = r.abs().amax(1, keepdim=True).clamp(min=1e-10) / top
    q = (r / s).round().clamp(-top, top)
    return (_pack(q).view(torch.int8), s[:, 0]) if fmt == "w4a4row" else (q.to(torch.int8), s)
