"""The measured workloads: what a program built on kea_kernels asks of it, through its public entry points.

Six kinds of call, each with its own range of sizes (see `draw`):
  linear     Int8MmaParts layer .linear: 1-bit weights, 1..3 activation parts, f32 / f16 rows in, f32 / f16 / bf16 out
  project    the projection provider (BinaryProjection through PartCount) with the LayerNorm and SiLU it fuses
  ternary    PackedLinear / PackedPointwiseConv1d: 2-bit weights, rows or a [B, K, T] convolution input
  grouped    lowbit.quantize + lowbit.gemm with one weight scale per 64 / 128 / 256 inputs
  attention  FastConformerEncoder.attention: relative-position self-attention of one layer
  frontend   the log-mel preprocessor and the x8 convolutional subsampling, audio to encoder input
  encoder    EncoderGraph: audio to encoder output, 24 layers, as a serving loop replays it

Matrix shapes are the encoder's own (1024 <-> 4096, 1024 -> 1024 / 2048 / 3072) and the decoder's (640 -> 2560,
640 -> 1030), and odd ones; row counts are frames (12.5 a second after subsampling) times clips.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch
import torch.nn.functional as F

_PACKAGE = str(Path(__file__).resolve().parents[1] / "kea-kernels_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
SHAPES = [(4096, 1024), (1024, 4096), (1024, 1024), (2048, 1024), (3072, 1024), (2560, 640), (1030, 640)]  # (n, k)
RATE, HOP, MELS, CHANNELS, D, HEADS, FF, TAPS, NFFT, WIN = 16000, 160, 128, 256, 1024, 8, 4096, 9, 512, 400
NORMS = ("norm_feed_forward1", "norm_self_att", "norm_conv", "norm_feed_forward2", "norm_out")
LINEARS = {"feed_forward1.linear1": (FF, D), "feed_forward1.linear2": (D, FF), "feed_forward2.linear1": (FF, D),
           "feed_forward2.linear2": (D, FF), "self_attn.linear_q": (D, D), "self_attn.linear_k": (D, D),
           "self_attn.linear_v": (D, D), "self_attn.linear_out": (D, D), "self_attn.linear_pos": (D, D),
           "conv.pointwise_conv1": (2 * D, D), "conv.pointwise_conv2": (D, D)}


# --- the cases -------------------------------------------------------------------------------------------------------

def listed() -> list[dict]:
    return [
        # one decoder step: a single token row through the joint projection (odd N); launches and host work only
        {"name": "decoder_row", "kind": "linear", "m": 1, "n": 1030, "k": 640, "parts": 1, "x": "f16", "y": "f16",
         "bias": True},
        # a 10-second clip's rows through an up projection, half precision in and out (the headline GEMM's shape)
        {"name": "linear_128", "kind": "linear", "m": 128, "n": 4096, "k": 1024, "parts": 1, "x": "f16", "y": "f16",
         "bias": False},
        # a ternary down projection with one scale per 128 inputs, one clip
        {"name": "grouped_128", "kind": "grouped", "m": 128, "n": 1024, "k": 4096, "parts": 1, "x": "f16", "y": "f16",
         "group": 128},
        # eight clips through LayerNorm + up projection + SiLU, the provider call an encoder makes
        {"name": "project_up_1000", "kind": "project", "m": 1000, "n": 4096, "k": 1024, "parts": 1, "norm": True,
         "silu": True},
        # a 30-second clip's down projection at three activation parts (full FP32 accuracy)
        {"name": "project_down_375_x3", "kind": "project", "m": 375, "n": 1024, "k": 4096, "parts": 3, "norm": False,
         "silu": False},
        # a ternary pointwise convolution on eight 30-second clips, channels-first input, two parts
        {"name": "ternary_conv_8x375_x2", "kind": "ternary", "batch": 8, "m": 3000, "n": 2048, "k": 1024, "parts": 2,
         "conv": True, "bias": True},
        # offline transcription: 128 ten-second clips' rows in one call
        {"name": "linear_16000", "kind": "linear", "m": 16000, "n": 4096, "k": 1024, "parts": 1, "x": "f16",
         "y": "f16", "bias": False},
        # one layer's attention on eight ten-second clips, and on two one-minute clips
        {"name": "attention_8x125", "kind": "attention", "batch": 8, "t": 125},
        {"name": "attention_2x750", "kind": "attention", "batch": 2, "t": 750},
        # audio to encoder input, eight ten-second clips
        {"name": "frontend_8x10s", "kind": "frontend", "batch": 8, "samples": 160000},
        # the whole encoder: one clip at two parts (interactive use), eight clips at three (batch use, full accuracy);
        # at one part 24 layers of 8-bit rounding decisions make any two roundings differ by 3e-2, so its GEMMs and
        # quantizers are measured layer by layer above
        {"name": "encoder_1x10s_x2", "kind": "encoder", "batch": 1, "samples": 160000, "parts": 2},
        {"name": "encoder_8x10s_x3", "kind": "encoder", "batch": 8, "samples": 160000, "parts": 3},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    """One case of the listed ranges: every kind, rows from 1 to 16000, clips from 1 to 60 seconds (the encoder and its
    graph up to 20), odd sizes throughout."""
    kind = rng.choice(["linear", "linear", "project", "project", "ternary", "grouped", "attention", "attention",
                       "frontend", "encoder"])
    if kind == "attention":
        batch = rng.choice([1, 1, 2, 3, 4, 8])
        return {"kind": kind, "batch": batch, "t": min(_log_int(rng, 12, 1000), math.isqrt(8 * 750 * 750 // batch))}
    if kind in ("frontend", "encoder"):
        batch = rng.choice([1, 1, 2, 3, 5, 8])
        seconds = min(math.exp(rng.uniform(0.0, math.log(60 if kind == "frontend" else 20))), 80 / batch)
        case = {"kind": kind, "batch": batch, "samples": max(RATE, int(seconds * RATE) - rng.randrange(HOP))}
        return dict(case, parts=rng.choice([2, 3])) if kind == "encoder" else case
    n, k = rng.choice(SHAPES)
    if rng.random() < 0.3:
        n, k = _log_int(rng, 200, 4096), _log_int(rng, 256, 4096)
    parts = rng.choice([1, 1, 2, 3])
    m = _log_int(rng, 1, 16000)
    m = max(1, min(m, 16000 * 1024 * 4096 // (n * k * parts)))
    case = {"kind": kind, "m": m, "n": n, "k": k, "parts": parts}
    if kind == "linear":
        case.update(x=rng.choice(["f32", "f16"]), y=rng.choice(["f32", "f16", "bf16"]), bias=rng.random() < 0.5)
    elif kind == "project":
        case.update(norm=rng.random() < 0.5, silu=rng.random() < 0.5)
    elif kind == "ternary":
        conv = rng.random() < 0.4
        batch = rng.choice([1, 2, 4, 8]) if conv else 1
        case.update(conv=conv, batch=batch, m=max(1, m // batch) * batch, bias=rng.random() < 0.5)
    else:
        # whole groups of 128, as grouped exports have, up to the rows an encoder call has
        case.update(n=-(-n // 16) * 16, k=-(-k // 128) * 128, m=min(m, 4000), group=rng.choice([64, 128, 256]),
                    x=rng.choice(["f32", "f16"]), y=rng.choice(["f32", "f16"]))
    return case


# --- inputs ----------------------------------------------------------------------------------------------------------

def _generator(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device="cuda") * std


def _rows(g, m: int, k: int) -> torch.Tensor:
    """Activation rows: normal, with row gains and a few large channels, as residual streams have."""
    x = _randn(g, m, k) * torch.exp(_randn(g, m, 1, std=0.3))
    return x * torch.where(torch.rand(k, generator=g, device="cuda") < 0.01, 6.0, 1.0)


def _scales(g, n: int, k: int) -> torch.Tensor:
    return (torch.rand(n, generator=g, device="cuda") + 0.5) / math.sqrt(k)


def _weights(g, n: int, k: int, bits: int) -> torch.Tensor:
    """int8 [n, k] signs (bits = 1) or ternary values (bits = 2)."""
    w = torch.randint(0, bits + 1, (n, k), generator=g, device="cuda", dtype=torch.int8)
    return 2 * w - 1 if bits == 1 else w - 1


def _pack(w: torch.Tensor, bits: int) -> torch.Tensor:
    """Export codes uint8 [n, ceil(k * bits / 8)]: a set bit is +1; 2-bit codes 0, 1, 2 are 0, +1, -1."""
    per = 8 // bits
    code = (w > 0).to(torch.uint8) if bits == 1 else torch.where(w < 0, 2, w).to(torch.uint8)
    code = F.pad(code, (0, -w.shape[1] % per)).view(w.shape[0], -1, per)
    shift = torch.arange(per, device=w.device, dtype=torch.uint8) * bits
    return (code << shift).sum(-1, dtype=torch.uint8)


def _matrix_inputs(case: dict, seed: int) -> dict:
    g = _generator(seed)
    m, n, k, kind = case["m"], case["n"], case["k"], case["kind"]
    bits = 1 if kind in ("linear", "project") else 2
    d = {"bits": bits, "w": _weights(g, n, k, bits), "scale": _scales(g, n, k), "bias": None, "norm": None}
    if case.get("bias"):
        d["bias"] = _randn(g, n, std=0.1)
    if case.get("norm"):
        d["norm"] = (1.0 + _randn(g, k, std=0.1), _randn(g, k, std=0.05))
    if kind == "grouped":
        groups = -(-k // case["group"])
        d["scale"] = (d["scale"][:, None] * (torch.rand(n, groups, generator=g, device="cuda") + 0.5)).half()
    d["x"] = _rows(g, m, k).to(DTYPES[case.get("x", "f32")])
    if case.get("conv"):
        d["x"] = d["x"].view(case["batch"], -1, k).transpose(1, 2).contiguous()
    return d


def _encoder_weights(seed: int, layers: int) -> dict:
    """Random parameters of the encoder under its checkpoint names, on the CPU."""
    g, bits = torch.Generator().manual_seed(seed), np.random.default_rng(seed)
    w = {}

    def randn(*shape, std=1.0):
        return torch.randn(*shape, generator=g) * std

    for i in range(layers):
        p = f"encoder.layers.{i}."
        for name, (n, k) in LINEARS.items():
            codes = np.frombuffer(bits.bytes(n * k // 8), np.uint8).reshape(n, k // 8).copy()
            w[p + name + ".codes"] = torch.from_numpy(codes)
            w[p + name + ".scale"] = (torch.rand(n, generator=g) + 0.5) / math.sqrt(k)
        for name in NORMS:
            w[p + name + ".weight"], w[p + name + ".bias"] = 1.0 + randn(D, std=0.05), randn(D, std=0.02)
        for name in ("pos_bias_u", "pos_bias_v"):
            w[p + "self_attn." + name] = randn(HEADS, D // HEADS, std=0.02)
        w[p + "conv.depthwise_conv.weight"] = randn(D, 1, TAPS, std=1 / 3)
        p += "conv.batch_norm."
        w[p + "weight"], w[p + "bias"] = 1.0 + randn(D, std=0.05), randn(D, std=0.02)
        w[p + "running_mean"], w[p + "running_var"] = randn(D, std=0.1), 1.0 + torch.rand(D, generator=g)
    p, c = "encoder.pre_encode.", CHANNELS
    for i in (0, 2, 5):
        w[p + f"conv.{i}.weight"], w[p + f"conv.{i}.bias"] = randn(c, 1, 3, 3, std=1 / 3), randn(c, std=0.02)
    for i in (3, 6):
        w[p + f"conv.{i}.weight"] = randn(c, c, 1, 1, std=1 / math.sqrt(c))
        w[p + f"conv.{i}.bias"] = randn(c, std=0.02)
    wide = c * (MELS // 8)
    w[p + "out.weight"], w[p + "out.bias"] = randn(D, wide, std=1 / math.sqrt(wide)), randn(D, std=0.02)
    return w


def _audio(case: dict, seed: int) -> torch.Tensor:
    """Noise with a slow envelope and a gliding tone: energy in every mel band, levels that change over time."""
    g, (b, s) = _generator(seed), (case["batch"], case["samples"])
    t = torch.arange(s, device="cuda", dtype=torch.float32) / RATE
    phase, rate = torch.rand(b, 1, generator=g, device="cuda"), 1.0 + torch.rand(b, 1, generator=g, device="cuda")
    envelope = 0.55 + 0.45 * torch.sin(2 * math.pi * (rate * t + phase))
    tone = torch.sin(2 * math.pi * (200 + 300 * torch.sin(0.7 * t + 6 * phase)) * t)
    return 0.1 * envelope * (_randn(g, b, s) + tone)


def _attention_inputs(case: dict, seed: int) -> tuple:
    g, (b, t) = _generator(seed), (case["batch"], case["t"])
    return (_randn(g, b, t, 3 * D), _randn(g, 2 * t - 1, D, std=0.7), _randn(g, HEADS, D // HEADS, std=0.1),
            _randn(g, HEADS, D // HEADS, std=0.1))


# --- the calls -------------------------------------------------------------------------------------------------------

def prepare(case: dict, seed: int) -> dict:
    from kea_kernels import encoder, lowbit
    from kea_kernels.binary import kernels, layer_parts, provider
    from kea_kernels.ternary import runtime

    kind, device = case["kind"], torch.device("cuda", 0)
    if kind in ("attention", "frontend", "encoder"):
        layers = 24 if kind == "encoder" else 1
        model = encoder.FastConformerEncoder(_encoder_weights(seed, layers), encoder.EncoderConfig(layers=layers),
                                             device, parts=case.get("parts", 1))
        if kind == "attention":
            return {"call": model.attention, "args": _attention_inputs(case, seed)}
        if kind == "frontend":
            return {"call": lambda audio: _frontend(model, audio), "args": (_audio(case, seed),)}
        graph = encoder.EncoderGraph(model, case["batch"], case["samples"])
        return {"call": graph, "args": (_audio(case, seed),)}

    d = _matrix_inputs(case, seed)
    m, n, k, parts, x, bits = case["m"], case["n"], case["k"], case["parts"], d["x"], d["bits"]
    codes = _pack(d["w"], bits)
    if kind == "linear":
        layer = layer_parts.LAYERS[parts].prepare(codes, d["scale"], d["bias"], k, device)
        return {"call": lambda x: layer.linear(x, out_dtype=DTYPES[case["y"]]), "args": (x,)}
    if kind == "project":
        table, modules = provider.prepare_table({"w": (codes, d["scale"], None, "linear", k)},
                                                layer_parts.LAYERS[parts], device)
        project = provider.PartCount(provider.BinaryProjection(table), parts)
        norm = None
        if d["norm"]:
            norm = torch.nn.LayerNorm(k, device=device).requires_grad_(False)
            norm.weight.copy_(d["norm"][0])
            norm.bias.copy_(d["norm"][1])
        act = "silu" if case["silu"] else ""
        return {"call": lambda x: project(x, modules["w"], False, parts, act, norm, None, ""), "args": (x,)}
    if kind == "ternary":
        cls = runtime.PackedPointwiseConv1d if case["conv"] else runtime.PackedLinear
        return {"call": cls(codes, d["scale"], k, d["bias"], mode=f"x{parts}"), "args": (x,)}
    words, scale = kernels.relayout_codes(codes, k, 2).to(device), d["scale"]

    def grouped(x):
        q, qs, _ = lowbit.quantize(x, (0, x.stride(0), x.stride(1), m), m, k, parts, qs_dtype=torch.float16)
        y = torch.empty(m, n, dtype=DTYPES[case["y"]], device=x.device)
        lowbit.gemm(2, q, qs, words, n, k, scale, None, y, ws_group=case["group"])
        return y

    return {"call": grouped, "args": (x,)}


def _frontend(model, audio):
    features = model.pre(audio)
    return features, model.subsample(features)


def run(state: dict):
    with torch.no_grad():
        return state["call"](*state["args"])


# --- what a pass cannot do without -----------------------------------------------------------------------------------

def _frames(case: dict) -> tuple[int, int]:
    """(feature frames, encoder frames) of a clip."""
    frames = t = case["samples"] // HOP
    for _ in range(3):
        t = (t - 1) // 2 + 1
    return frames, t


def _attention_flops(b: int, t: int) -> int:
    return 2 * b * t * t * D * 3


def _frontend_work(case: dict) -> tuple[int, int]:
    b, (frames, t) = case["batch"], _frames(case)
    c, f = CHANNELS, MELS
    flops = b * frames * (5 * NFFT * 9 // 2 + 2 * NFFT)
    flops += 2 * b * c * ((frames // 2) * (f // 2) * 9 + (frames // 4) * (f // 4) * (9 + c) + t * (f // 8) * (9 + c))
    flops += 2 * b * t * c * (f // 8) * D
    weights = 4 * (2 * c * c + 30 * c + (c * (f // 8) + 1) * D)
    return 4 * b * (case["samples"] + frames * MELS + t * D) + weights, flops


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "attention":
        b, t = case["batch"], case["t"]
        return {"bytes": 4 * (b * t * 4 * D + (2 * t - 1) * D), "flops": _attention_flops(b, t)}
    if kind in ("frontend", "encoder"):
        nbytes, flops = _frontend_work(case)
        if kind == "encoder":
            b, (_, t) = case["batch"], _frames(case)
            size = sum(n * k for name, (n, k) in LINEARS.items() if not name.endswith("linear_pos"))
            flops += 24 * (2 * b * t * size * case["parts"] + _attention_flops(b, t) + 2 * b * t * D * TAPS)
            nbytes += 24 * (size // 8 + 4 * (2 * t - 1) * D) - 4 * b * _frames(case)[0] * MELS
        return {"bytes": nbytes, "flops": flops}
    m, n, k = case["m"], case["n"], case["k"]
    size = {"f32": 4, "f16": 2, "bf16": 2}
    bits = 1 if kind in ("linear", "project") else 2
    nbytes = m * k * size[case.get("x", "f32")] + m * n * size[case.get("y", "f32")] + n * -(-k * bits // 8)
    nbytes += 2 * n * -(-k // case["group"]) if kind == "grouped" else 4 * n
    nbytes += 4 * n * bool(case.get("bias")) + 8 * k * bool(case.get("norm"))
    return {"bytes": nbytes, "flops": 2 * m * n * k * case["parts"]}


# --- how close another correct implementation comes ------------------------------------------------------------------

def tolerance(case: dict) -> dict:
    """Relative to the result. One activation part is an 8-bit rounding: an input that another rounding of the
    LayerNorm or scale moves across a rounding boundary changes by a whole step, which shows as 1e-4 or so of a row."""
    kind = case["kind"]
    if kind == "attention":
        return {"rel": 3e-6, "max": 2e-4}
    if kind == "frontend":
        return {"rel": 1e-5, "max": 1e-3}
    if kind == "encoder":
        return {2: {"rel": 3e-4, "max": 2e-3}, 3: {"rel": 2e-6, "max": 2e-5}}[case["parts"]]
    out = {"f32": 1e-6, "f16": 1e-3, "bf16": 8e-3}[case.get("y", "f32")]
    return {"rel": max(out, {1: 2e-3, 2: 1e-5, 3: 1e-6}[case["parts"]]), "max": 0.05}


# --- the same results in 64 bits -------------------------------------------------------------------------------------

def _layer_norm64(z, w, b):
    return F.layer_norm(z, (z.shape[-1],), w.double(), b.double(), 1e-5)


def _parts64(z: torch.Tensor, parts: int, half_scales: bool = False) -> torch.Tensor:
    """The value that the residual int8 parts of each row stand for: s = max|z| / 127, q = round(z / s), z -= q s."""
    total = torch.zeros_like(z)
    for _ in range(parts):
        s = (z.abs().amax(-1, keepdim=True) / 127).clamp_min(1e-30)
        if half_scales:
            s = s.half().double().clamp(2.0 ** -24, 65504.0)
        part = torch.round(z / s).clamp(-127, 127) * s
        total += part
        z = z - part
    return total


def _linear64(z, codes: torch.Tensor, scale, parts: int) -> torch.Tensor:
    shift = torch.arange(8, device=z.device, dtype=torch.uint8)
    bits = (codes.to(z.device)[:, :, None] >> shift) & 1
    w = bits.view(codes.shape[0], -1).double() * 2 - 1
    return (_parts64(z, parts) @ w.t()) * scale.to(z.device).double()


def _attention64(qkv, pos, u, v):
    b, t, _ = qkv.shape
    dk = D // HEADS
    q, k, val = (x.transpose(1, 2).contiguous() for x in qkv.double().view(b, t, 3, HEADS, dk).unbind(2))
    p = pos.double().view(2 * t - 1, HEADS, dk).permute(1, 2, 0).contiguous()
    content = (q + u.double()[:, None]) @ k.transpose(2, 3).contiguous()
    band = (q + v.double()[:, None]) @ p
    i = torch.arange(t, device=qkv.device)
    index = (t - 1 - i[:, None] + i[None, :]).expand(b, HEADS, t, t)
    a = torch.softmax((content + band.gather(3, index)) / math.sqrt(dk), -1)
    return (a @ val).transpose(1, 2).reshape(b, t, D)


def _mel_filters64() -> torch.Tensor:
    """[MELS, bins] triangular filters on the Slaney mel scale with area normalisation."""
    def to_mel(f):
        return np.where(f >= 1000, 15 + 27 * np.log(np.maximum(f, 1e-10) / 1000) / math.log(6.4), f * 3 / 200)

    def to_hz(m):
        return np.where(m >= 15, 1000 * np.exp(math.log(6.4) / 27 * (m - 15)), m * 200 / 3)

    freqs = np.linspace(0, RATE / 2, NFFT // 2 + 1)
    edges = to_hz(np.linspace(to_mel(np.float64(0)), to_mel(np.float64(RATE / 2)), MELS + 2))
    low, mid, high = edges[:-2, None], edges[1:-1, None], edges[2:, None]
    tri = np.maximum(0, np.minimum((freqs - low) / (mid - low), (high - freqs) / (high - mid)))
    return torch.from_numpy(tri * 2 / (high - low)).cuda()


def _features64(audio: torch.Tensor) -> torch.Tensor:
    a = audio.double()
    a = torch.cat([a[:, :1], a[:, 1:] - 0.97 * a[:, :-1]], 1)
    frames = F.pad(a, (NFFT // 2, NFFT // 2)).unfold(1, NFFT, HOP)[:, :audio.shape[1] // HOP]
    window = F.pad(torch.hann_window(WIN, periodic=False, dtype=torch.float64, device="cuda"),
                   ((NFFT - WIN) // 2, (NFFT - WIN + 1) // 2))
    power = torch.fft.rfft(frames * window).abs().square()                  # [B, frames, bins]
    mel = torch.log((power @ _mel_filters64().t().contiguous()).transpose(1, 2) + 2.0 ** -24)
    return (mel - mel.mean(2, keepdim=True)) / (mel.std(2, keepdim=True) + 1e-5)


def _taps64(x, w, b):
    """3x3 / stride 2 / padding 1, one filter per output channel, x [B, 1 or C, T, F]."""
    x, w = F.pad(x, (1, 1, 1, 1)), w.double()
    t, f = (x.shape[2] - 3) // 2 + 1, (x.shape[3] - 3) // 2 + 1
    y = b.double()[:, None, None].expand(x.shape[0], -1, t, f).clone()
    for i in range(3):
        for j in range(3):
            y += w[:, 0, i, j][:, None, None] * x[:, :, i:i + 2 * t - 1:2, j:j + 2 * f - 1:2]
    return y


def _subsample64(features, w: dict) -> torch.Tensor:
    s = {name[len("encoder.pre_encode."):]: v.cuda() for name, v in w.items() if "pre_encode" in name}
    outs = []
    for clip in features.double().transpose(1, 2)[:, None, None]:           # a clip at a time: [1, 1, frames, mels]
        x = F.relu(_taps64(clip, s["conv.0.weight"], s["conv.0.bias"]))
        for i in (2, 5):
            x = _taps64(x, s[f"conv.{i}.weight"], s[f"conv.{i}.bias"])
            c, (t, f) = x.shape[1], x.shape[2:]
            x = s[f"conv.{i + 1}.weight"].double().view(c, c) @ x.view(c, t * f)
            x = F.relu(x + s[f"conv.{i + 1}.bias"].double()[:, None]).view(1, c, t, f)
        outs.append(x[0].transpose(0, 1).reshape(t, c * f) @ s["out.weight"].double().t().contiguous())
    return (torch.stack(outs) + s["out.bias"].double()) * math.sqrt(D)


def _encoder64(audio, w: dict, parts: int) -> torch.Tensor:
    x = _subsample64(_features64(audio), w)
    b, t, _ = x.shape
    # the sinusoids are inputs of the projection, in 32 bits as the model makes them
    place = torch.arange(t - 1, -t, -1, dtype=torch.float32, device="cuda")[:, None]
    rate = torch.exp(torch.arange(0, D, 2, dtype=torch.float32, device="cuda") * (-math.log(10000.0) / D))
    pe = torch.stack([torch.sin(place * rate), torch.cos(place * rate)], -1).view(2 * t - 1, D).double()
    for i in range(24):
        p = f"encoder.layers.{i}."
        lw = {name[len(p):]: v.cuda() for name, v in w.items() if name.startswith(p)}

        def linear(name, z):
            return _linear64(z, lw[name + ".codes"], lw[name + ".scale"], parts)

        def norm(name, z):
            return _layer_norm64(z, lw[name + ".weight"], lw[name + ".bias"])

        def ff(name, z):
            return linear(name + ".linear2", F.silu(linear(name + ".linear1", z)))

        x = x + 0.5 * ff("feed_forward1", norm("norm_feed_forward1", x))
        z = norm("norm_self_att", x)
        qkv = torch.cat([linear("self_attn.linear_" + c, z) for c in "qkv"], -1)
        a = _attention64(qkv, linear("self_attn.linear_pos", pe), lw["self_attn.pos_bias_u"], lw["self_attn.pos_bias_v"])
        x = x + linear("self_attn.linear_out", a)
        z = F.glu(linear("conv.pointwise_conv1", norm("norm_conv", x)), -1)
        bn = {key: lw["conv.batch_norm." + key].double() for key in ("weight", "bias", "running_mean", "running_var")}
        gain = bn["weight"] / torch.sqrt(bn["running_var"] + 1e-5)
        taps = lw["conv.depthwise_conv.weight"].double()[:, 0] * gain[:, None]
        padded = F.pad(z, (0, 0, TAPS // 2, TAPS // 2))
        z = sum(padded[:, j:j + t] * taps[:, j] for j in range(TAPS)) + bn["bias"] - bn["running_mean"] * gain
        x = x + linear("conv.pointwise_conv2", F.silu(z))
        x = x + 0.5 * ff("feed_forward2", norm("norm_feed_forward2", x))
        x = norm("norm_out", x)
    return x


@torch.no_grad()
def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "attention":
        return _attention64(*_attention_inputs(case, seed))
    if kind == "frontend":
        features = _features64(_audio(case, seed))
        return features, _subsample64(features, _encoder_weights(seed, 1))
    if kind == "encoder":
        return _encoder64(_audio(case, seed), _encoder_weights(seed, 24), case["parts"])
    d = _matrix_inputs(case, seed)
    z = d["x"].double()
    z = z.transpose(1, 2) if case.get("conv") else z
    if d["norm"]:
        z = _layer_norm64(z, *d["norm"])
    w = d["w"].double()
    if kind == "grouped":
        w = w * d["scale"].double().repeat_interleave(case["group"], 1)[:, :w.shape[1]]
    else:
        w = w * d["scale"].double()[:, None]
    y = _parts64(z, case["parts"], kind == "grouped") @ w.t().contiguous()
    if d["bias"] is not None:
        y = y + d["bias"].double()
    if case.get("silu"):
        y = F.silu(y)
    return y.transpose(1, 2) if case.get("conv") else y
