"""The decode stage's work as its users have it done, one case per kind and size of call: whole
decodes through the codec, vocoder and graph-runner entry points, and the single blocks and layers
that callers reach through ``sglang_omni_amd.kernels`` and ``sglang_omni_amd.utils``.

``prepare`` makes what a program holds before the call (weights, slot pool, inputs; everything
from the seed), ``run`` is one call, ``exact`` the same result in float64 from plain torch. The
networks are the repository's own configurations with random weights: kaiming-scaled convs with
small biases (bf16 values, as a checkpoint holds them) and Snake frequencies around one.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path
from types import SimpleNamespace

import torch

sys.path.insert(1, str(Path.cwd() / "sglang-omni_amd"))

from sglang_omni_amd import _native as N  # noqa: E402
from sglang_omni_amd.kernels import (  # noqa: E402
    ResidualUnitWeights,
    SnakeBetaCoefficients,
    fused_bias_snake_beta,
    fused_conv,
    pack_conv1d,
    residual_stack,
    rvq_gather_sum,
)
from sglang_omni_amd.kernels import code2wav_front as front  # noqa: E402
from sglang_omni_amd.kernels.conv import FinalConv, stack_coefficients  # noqa: E402
from sglang_omni_amd.kernels.gemm import (  # noqa: E402
    SCALED_RESIDUAL,
    linear,
    linear_rope_kv,
    pack_linear,
)
from sglang_omni_amd.kernels.hift import HiftStft  # noqa: E402
from sglang_omni_amd.models import (  # noqa: E402
    CODEC_24K,
    HIFIGAN_24K,
    QWEN3_CODE2WAV,
    CodecGraphRunner,
    DacCodecDecoder,
    GraphKey,
    HifiGanVocoder,
)
from sglang_omni_amd.utils.channels_last_conv import (  # noqa: E402
    channels_last_conv1d,
    channels_last_conv_transpose1d,
    channels_last_weight,
)

DEVICE = torch.device("cuda", 0)
BF16, F16, F32, F64 = torch.bfloat16, torch.float16, torch.float32, torch.float64
DTYPES = {"bf16": BF16, "f16": F16, "f32": F32}
# a ConvTranspose1d of the vocoder per stage: (channels in, channels out, kernel, stride)
UPSAMPLERS = ((512, 256, 16, 8), (256, 128, 11, 5), (128, 64, 7, 3), (64, 32, 8, 4))


def listed() -> list[dict]:
    return [
        # one listener: the next four frames of a single stream, replayed from the graph a serving
        # loop captures for it (the smallest step, all launches and latency)
        {"name": "stream 1x4", "kind": "stream", "streams": 1, "frames": 4, "graph": True},
        # a loaded server's step: the next 12-frame chunk of 64 streams, state in the slot pool
        {"name": "stream 64x12", "kind": "stream", "streams": 64, "frames": 12, "graph": False},
        # one finished utterance of 20 s decoded whole
        {"name": "utterance 1x250", "kind": "utterance", "rows": 1, "frames": 250},
        # a mel vocoder batch: 16 clips of 10 s
        {"name": "hifigan 16x500", "kind": "hifigan", "rows": 16, "frames": 500},
        # a 192-channel residual unit as the decoders launch it, rows of an odd length
        {"name": "unit192 12x5003", "kind": "unit", "rows": 12, "samples": 5003, "channels": 192,
         "dilation": 9},
        # the last block's three residual units and the output conv, E4M3 weights (the long-form
        # decoder's option), rows of an odd length
        {"name": "stack fp8 8x60001", "kind": "stack", "rows": 8, "samples": 60001, "fp8": True},
        # a code2wav transformer layer while streaming: five new frames of 16 streams, K / V rings
        {"name": "layer decode 16x5", "kind": "layer", "rows": 16, "frames": 5, "warm": True},
        # the same layer over whole utterances
        {"name": "layer prefill 4x301", "kind": "layer", "rows": 4, "frames": 301, "warm": False},
        # the vocoder's transforms at its output rate: source spectrum and inverse tail, 16 x 10 s
        {"name": "hift 16x240000", "kind": "hift", "rows": 16, "samples": 240000},
        # a residual unit through the channels-last conv and Snake functions in half precision,
        # as a caller of those functions runs its decoder
        {"name": "channels-last unit f16", "kind": "cl_unit", "rows": 4, "samples": 4801,
         "channels": 192, "dilation": 3, "dtype": "f16"},
        # a float32 vocoder upsampler through the same functions
        {"name": "channels-last up f32", "kind": "cl_up", "rows": 2, "samples": 2003, "stage": 1,
         "dtype": "f32"},
        # dequantizing a long batch: 32 codebooks, 8 x 120 s
        {"name": "rvq 8x1500", "kind": "rvq", "rows": 8, "frames": 1500, "books": 32,
         "entries": 1024, "codes": "i32", "tables": "bf16"},
    ]


def _log(rng, low: int, high: int) -> int:
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high + 0.5))))))


def draw(rng) -> dict:
    kind = rng.choice(["stream", "stream", "utterance", "hifigan", "unit", "stack", "layer", "hift",
                       "cl_unit", "cl_up", "rvq"])
    if kind == "stream":
        streams = _log(rng, 1, 64)
        return {"kind": kind, "streams": streams, "frames": rng.randint(1, 12),
                "graph": streams <= 8}
    if kind == "utterance":
        rows = rng.randint(1, 4)
        return {"kind": kind, "rows": rows, "frames": _log(rng, 20, 1000 // rows)}
    if kind == "hifigan":
        return {"kind": kind, "rows": _log(rng, 1, 16), "frames": _log(rng, 30, 500)}
    if kind == "unit":
        rows = _log(rng, 1, 16)
        channels = rng.choice([192, 384, 768])
        return {"kind": kind, "rows": rows, "channels": channels, "dilation": rng.choice([1, 3, 9]),
                "samples": _log(rng, 960, 120000 * 192 // channels // rows)}
    if kind == "stack":
        rows = _log(rng, 1, 16)
        return {"kind": kind, "rows": rows, "samples": _log(rng, 1920, 480000 // rows),
                "fp8": rng.random() < 0.5}
    if kind == "layer":
        warm = rng.random() < 0.6
        rows = _log(rng, 1, 64 if warm else 8)
        return {"kind": kind, "rows": rows, "warm": warm,
                "frames": rng.randint(1, 12) if warm else _log(rng, 13, 1204 // rows)}
    if kind == "hift":
        return {"kind": kind, "rows": _log(rng, 1, 16), "samples": 4 * _log(rng, 600, 60000)}
    if kind == "cl_unit":
        channels = rng.choice([96, 192, 384])
        rows = rng.randint(1, 4)
        return {"kind": kind, "rows": rows, "channels": channels, "dilation": rng.choice([1, 3, 9]),
                "samples": _log(rng, 100, 19204 * 192 * 192 // (channels * channels) // rows),
                "dtype": rng.choice(["f16", "f16", "bf16"])}
    if kind == "cl_up":
        rows, stage = rng.randint(1, 2), rng.randrange(4)
        return {"kind": kind, "rows": rows, "stage": stage,
                "samples": _log(rng, 50, 500 * 4 ** stage // rows),
                "dtype": rng.choice(["f32", "f32", "f16", "bf16"])}
    return {"kind": kind, "rows": _log(rng, 1, 64), "frames": _log(rng, 2, 187),
            "books": rng.choice([8, 16, 32]), "entries": rng.choice([1024, 2048]),
            "codes": rng.choice(["i32", "i64"]), "tables": rng.choice(["bf16", "f32"])}


# ------------------------------------------------------------------ weights and inputs


class _Random:
    """Seeded draws on the GPU."""

    def __init__(self, seed: int):
        self.gen = torch.Generator(device=DEVICE).manual_seed(seed)

    def normal(self, *shape: int, std: float = 1.0) -> torch.Tensor:
        return torch.randn(*shape, generator=self.gen, device=DEVICE) * std

    def integers(self, high: int, *shape: int) -> torch.Tensor:
        return torch.randint(0, high, shape, generator=self.gen, device=DEVICE)

    def values(self, dtype: torch.dtype, *shape: int, std: float) -> torch.Tensor:
        """float32 normals that ``dtype`` holds exactly."""
        return self.normal(*shape, std=std).to(dtype).float()

    def conv(self, c_out: int, c_in: int, k: int, gain: float = 0.85, dtype=BF16) -> dict:
        return {"weight": self.values(dtype, c_out, c_in, k, std=gain / math.sqrt(c_in * k)),
                "bias": self.values(dtype, c_out, std=0.02)}

    def conv_transpose(self, c_in: int, c_out: int, k: int, gain: float = 0.85, dtype=BF16) -> dict:
        return {"weight": self.values(dtype, c_in, c_out, k, std=gain / math.sqrt(c_out * k)),
                "bias": self.values(dtype, c_out, std=0.02)}

    def snake(self, channels: int) -> torch.Tensor:
        return torch.exp(self.normal(channels, std=0.2))


def _codec_weights(r: _Random) -> dict:
    """The 24 kHz codec: 16 codebooks of 2048 x 512, 1536 channels, strides 8 / 8 / 5 / 6."""
    tree = {"codebooks": r.values(BF16, 16, 2048, 512, std=0.02), "in_conv": r.conv(1536, 512, 7),
            "blocks": []}
    c = 1536
    for stride in (8, 8, 5, 6):
        half = c // 2
        block = {"stride": stride, "alpha": r.snake(c),
                 "up": r.conv_transpose(c, half, 2 * stride), "units": []}
        for d in (1, 3, 9):
            block["units"].append({"dilation": d, "alpha1": r.snake(half),
                                   "conv1": r.conv(half, half, 7), "alpha2": r.snake(half),
                                   "conv2": r.conv(half, half, 1)})
        tree["blocks"].append(block)
        c = half
    tree["final"] = {"alpha": r.snake(c), "conv": r.conv(1, c, 7)}
    return tree


def _hifigan_weights(r: _Random) -> dict:
    """The mel vocoder: 80 mels, 512 channels, x480, ResBlocks of 3 / 7 / 11 taps."""
    tree = {"slope": 0.1, "final_slope": 0.01, "conv_pre": r.conv(512, 80, 7, 0.8), "stages": []}
    for c_in, c_out, k, rate in UPSAMPLERS:
        stage = {"rate": rate, "up": r.conv_transpose(c_in, c_out, k, 0.8), "resblocks": []}
        for taps in (3, 7, 11):
            stage["resblocks"].append({
                "kernel": taps, "dilations": (1, 3, 5),
                "convs1": [r.conv(c_out, c_out, taps, 0.8) for _ in range(3)],
                "convs2": [r.conv(c_out, c_out, taps, 0.8) for _ in range(3)]})
        tree["stages"].append(stage)
    tree["conv_post"] = r.conv(1, 32, 7, 0.8)
    return tree


def _quantized(node: dict, fp8: bool) -> dict:
    """A conv with its E4M3 weight and per-output-channel scale, as an fp8 checkpoint holds it."""
    if not fp8:
        return node
    w = node["weight"]
    scale = w.reshape(w.shape[0], -1).abs().amax(dim=1) / 448.0
    return {"weight": (w / scale[:, None, None]).to(torch.float8_e4m3fn), "weight_scale": scale,
            "bias": node["bias"]}


def _dense(node: dict) -> torch.Tensor:
    w = node["weight"].to(F64)
    return w * node["weight_scale"].to(F64)[:, None, None] if "weight_scale" in node else w


def _unit_weights(r: _Random, case: dict) -> SimpleNamespace:
    c = case["channels"]
    return SimpleNamespace(conv1=r.conv(c, c, 7), conv2=r.conv(c, c, 1), alpha1=r.snake(c),
                           alpha2=r.snake(c), alpha3=r.snake(c),
                           x=r.normal(case["rows"], case["samples"], c, std=0.5).to(F16))


def _stack_weights(r: _Random, case: dict) -> SimpleNamespace:
    units = [SimpleNamespace(dilation=d, alpha1=r.snake(96), alpha2=r.snake(96),
                             conv1=_quantized(r.conv(96, 96, 7), case["fp8"]),
                             conv2=_quantized(r.conv(96, 96, 1), case["fp8"])) for d in (1, 3, 9)]
    return SimpleNamespace(units=units, alpha=r.snake(96), final=r.conv(1, 96, 7, 0.3),
                           x=r.normal(case["rows"], case["samples"], 96, std=0.5).to(F16))


def _layer_weights(r: _Random, case: dict) -> SimpleNamespace:
    """A code2wav pre-transformer layer (1024 wide, 16 heads of 64, 3072 MLP, 72-frame window)
    and, while streaming, rings holding a full window of every stream's past."""
    rows, frames, ring = case["rows"], case["frames"], 71 + 64

    def lin(out: int, into: int) -> torch.Tensor:
        return r.values(BF16, out, into, std=1 / math.sqrt(into))

    w = SimpleNamespace(qkv=lin(3072, 1024), o=lin(1024, 1024), gate_up=lin(6144, 1024),
                        down=lin(1024, 3072), norm1=1 + r.normal(1024, std=0.1),
                        norm2=1 + r.normal(1024, std=0.1), scale1=r.normal(1024, std=0.5),
                        scale2=r.normal(1024, std=0.5),
                        h=r.normal(rows * frames, 1024), ring=ring)
    w.inv_freq = 1.0 / (10000.0 ** (torch.arange(0, 64, 2, dtype=F32, device=DEVICE) / 64))
    if case["warm"]:
        w.keys = r.normal(rows * ring, 1024).to(BF16)
        w.values = r.normal(rows * ring, 1024).to(BF16)
        w.positions = 72 + r.integers(2000, rows)
        w.slots = torch.randperm(rows, generator=r.gen, device=DEVICE)
    return w


def _hift_inputs(r: _Random, case: dict) -> tuple[torch.Tensor, torch.Tensor]:
    """A source waveform and the last conv's output (log magnitudes around e^-3, phases)."""
    rows, samples = case["rows"], case["samples"]
    h = r.normal(rows, samples // 4 + 1, 18, std=0.5)
    h[..., :9] -= 3.0
    return r.normal(rows, samples, std=0.1), h


def _cl_unit_weights(r: _Random, case: dict) -> SimpleNamespace:
    c, dt, d = case["channels"], DTYPES[case["dtype"]], case["dilation"]
    rows, samples = case["rows"], case["samples"]
    return SimpleNamespace(
        conv1=r.conv(c, c, 7, dtype=dt), conv2=r.conv(c, c, 1, dtype=dt),
        alpha1=r.values(dt, c, std=0.2), beta1=r.values(dt, c, std=0.2),
        alpha2=r.values(dt, c, std=0.2), beta2=r.values(dt, c, std=0.2),
        u=r.normal(rows, 6 * d + samples, c, std=0.5).to(dt), x=r.normal(rows, samples, c, std=0.5).to(dt))


def _cl_up_weights(r: _Random, case: dict) -> SimpleNamespace:
    c_in, c_out, k, stride = UPSAMPLERS[case["stage"]]
    dt = DTYPES[case["dtype"]]
    return SimpleNamespace(up=r.conv_transpose(c_in, c_out, k, dtype=dt), stride=stride,
                           padding=(k - stride) // 2,
                           x=r.normal(case["rows"], case["samples"], c_in, std=0.5).to(dt))


def _rvq_inputs(r: _Random, case: dict) -> tuple[torch.Tensor, torch.Tensor]:
    codes = r.integers(case["entries"], case["rows"], case["books"], case["frames"])
    tables = r.normal(case["books"], case["entries"], 512, std=0.02).to(DTYPES[case["tables"]])
    return codes.to(torch.int32 if case["codes"] == "i32" else torch.int64), tables


def _stream_codes(r: _Random, case: dict) -> torch.Tensor:
    """The chunk a step decodes and the one before it, which fills the streams' state."""
    return r.integers(2048, case["streams"], 16, 2 * case["frames"])


# ------------------------------------------------------------------ prepare


def _coefficients(alpha: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    return alpha, (alpha + 1e-9).reciprocal()


def _module(cls, node: dict, dtype: torch.dtype, **kw):
    c_out, c_in = node["weight"].shape[:2]
    if cls is torch.nn.ConvTranspose1d:
        c_out, c_in = c_in, c_out
    conv = cls(c_in, c_out, node["weight"].shape[2], device=DEVICE, dtype=dtype, **kw)
    with torch.no_grad():
        conv.weight.copy_(node["weight"])
        conv.bias.copy_(node["bias"])
    return conv.requires_grad_(False)


def prepare(case: dict, seed: int) -> SimpleNamespace:
    r = _Random(seed)
    kind = case["kind"]
    s = SimpleNamespace(kind=kind, case=case)
    if kind == "stream":
        s.decoder = DacCodecDecoder(_codec_weights(r), CODEC_24K, device=DEVICE)
        rows, frames = case["streams"], case["frames"]
        codes = _stream_codes(r, case)
        s.pool = s.decoder.new_state_pool(rows, capture_slots=rows if case["graph"] else 0)
        s.slots = s.pool.stage_index([s.pool.acquire() for _ in range(rows)])
        s.runner = None
        if case["graph"]:
            s.runner = CodecGraphRunner(s.decoder, s.pool, [GraphKey(rows, frames, "next")])
            failed = s.runner.capture_all()
            if failed:
                raise RuntimeError(f"the step's graph was not published: {failed}")
        s.decoder.decode_slots(codes[..., :frames].contiguous(), s.pool, s.slots, first_decode=True)
        s.codes = codes[..., frames:].contiguous()
    elif kind == "utterance":
        s.decoder = DacCodecDecoder(_codec_weights(r), CODEC_24K, device=DEVICE)
        s.codes = r.integers(2048, case["rows"], 16, case["frames"])
    elif kind == "hifigan":
        s.vocoder = HifiGanVocoder(_hifigan_weights(r), HIFIGAN_24K, device=DEVICE)
        s.mel = r.normal(case["rows"], 80, case["frames"], std=2.0) - 5.0
    elif kind == "unit":
        w = _unit_weights(r, case)
        s.conv1 = pack_conv1d(w.conv1["weight"], w.conv1["bias"], dilation=case["dilation"])
        s.conv2 = pack_conv1d(w.conv2["weight"], w.conv2["bias"])
        (a1, b1), s.mid, s.next = map(_coefficients, (w.alpha1, w.alpha2, w.alpha3))
        s.x = w.x
        s.u = (w.x.float() + b1 * torch.sin(a1 * w.x.float()) ** 2).to(BF16)
        s.out, s.h, s.sum = torch.empty_like(s.u), torch.empty_like(s.u), torch.empty_like(s.x)
    elif kind == "stack":
        w = _stack_weights(r, case)

        def pack(node, d=1):
            return pack_conv1d(node["weight"], node["bias"], dilation=d,
                               scale=node.get("weight_scale"))

        s.units = [ResidualUnitWeights(pack(u.conv1, u.dilation), pack(u.conv2),
                                       *_coefficients(u.alpha1), *_coefficients(u.alpha2))
                   for u in w.units]
        s.a, s.b = _coefficients(w.alpha)
        s.table = stack_coefficients(s.units, s.a, s.b)
        s.x = w.x
        s.final = FinalConv(w.final["weight"][0].t().contiguous(), w.final["bias"], N.ACT_TANH,
                            torch.empty(case["rows"], 1, case["samples"], device=DEVICE))
    elif kind == "layer":
        w = _layer_weights(r, case)
        s.w, m = w, case["rows"] * case["frames"]
        s.qkv_w, s.o_w, s.down_w = pack_linear(w.qkv), pack_linear(w.o), pack_linear(w.down)
        s.gate_up_w = pack_linear(w.gate_up, gated=True)
        s.normed, s.attn = (torch.empty(m, 1024, dtype=BF16, device=DEVICE) for _ in range(2))
        s.qkv, s.act = (torch.empty(m, 3072, dtype=BF16, device=DEVICE) for _ in range(2))
        s.h1, s.h2 = torch.empty_like(w.h), torch.empty_like(w.h)
        s.rings = {}
        if case["warm"]:
            s.rings = {"slot_index": w.slots, "positions": w.positions, "key_ring": w.keys,
                       "value_ring": w.values, "ring_frames": w.ring}
    elif kind == "hift":
        s.stft = HiftStft(torch.hann_window(16, periodic=True), 4, device=DEVICE)
        s.signal, s.h = _hift_inputs(r, case)
    elif kind == "cl_unit":
        w = _cl_unit_weights(r, case)
        dt = s.dtype = DTYPES[case["dtype"]]
        s.conv1 = _module(torch.nn.Conv1d, w.conv1, dt, dilation=case["dilation"])
        s.conv2 = _module(torch.nn.Conv1d, w.conv2, dt)
        s.w1, s.w2 = channels_last_weight(s.conv1), channels_last_weight(s.conv2)
        s.mid, s.next = (SnakeBetaCoefficients.from_activation(SimpleNamespace(
            alpha=a.to(dt), beta=b.to(dt), no_div_by_zero=1e-9))
            for a, b in ((w.alpha1, w.beta1), (w.alpha2, w.beta2)))
        s.u, s.x = w.u, w.x
    elif kind == "cl_up":
        w = _cl_up_weights(r, case)
        s.up = _module(torch.nn.ConvTranspose1d, w.up, DTYPES[case["dtype"]], stride=w.stride,
                       padding=w.padding)
        s.weight = channels_last_weight(s.up)
        s.x = w.x
    else:
        s.codes, s.tables = _rvq_inputs(r, case)
    return s


# ------------------------------------------------------------------ run


def run(s: SimpleNamespace):
    return _RUN[s.kind](s)


def _run_stream(s):
    if s.runner is not None:
        wave = s.runner.run(s.codes, s.slots, first_decode=False).output
    else:
        wave = s.decoder.decode_slots(s.codes, s.pool, s.slots, first_decode=False)
    return {"wave": wave, "parity": s.pool.parity, "histories": s.pool.histories}


def _run_unit(s):
    """The two convs of a unit as the decoders launch them: fused for 192 channels."""
    kw = dict(residual=s.x, sum_out=s.sum, activation=N.ACT_SNAKE, act_a=s.next[0], act_b=s.next[1])
    if s.case["channels"] == 192:
        fused_conv(s.u, s.conv1, s.out, second=s.conv2, mid_activation=N.ACT_SNAKE,
                   mid_a=s.mid[0], mid_b=s.mid[1], **kw)
    else:
        fused_conv(s.u, s.conv1, s.h, activation=N.ACT_SNAKE, act_a=s.mid[0], act_b=s.mid[1])
        fused_conv(s.h, s.conv2, s.out, **kw)
    return {"out": s.out, "sum": s.sum}


def _run_layer(s):
    w, batch = s.w, s.case["rows"]
    cold = not s.case["warm"]
    front.rms_norm_residual(w.h, w.norm1, 1e-5, s.normed)
    linear_rope_kv(s.normed, s.qkv_w, s.qkv, batch, 16, 16, 64, w.inv_freq, cold=cold, **s.rings)
    front.window_attention(s.qkv, batch, 16, 16, 64, 72, 0.125, s.attn, cold=cold, **s.rings)
    linear(s.attn, s.o_w, s.h1, epilogue=SCALED_RESIDUAL, scale=w.scale1, residual=w.h)
    front.rms_norm_residual(s.h1, w.norm2, 1e-5, s.normed)
    linear(s.normed, s.gate_up_w, s.act)
    linear(s.act, s.down_w, s.h2, epilogue=SCALED_RESIDUAL, scale=w.scale2, residual=s.h1)
    return {"h": s.h2, "qkv": s.qkv, **({} if cold else {"keys": w.keys, "values": w.values})}


def _run_cl_unit(s):
    length = s.x.shape[1]
    y = channels_last_conv1d(s.u, s.conv1, s.w1, None, length)[:, :length]
    h = torch.empty_like(y)
    fused_bias_snake_beta(y, s.conv1.bias, s.mid, h)
    z = channels_last_conv1d(h, s.conv2, s.w2, None, length)
    out, total = torch.empty_like(z), torch.empty_like(z)
    fused_bias_snake_beta(z, s.conv2.bias, s.next, out, residual=s.x, sum_out=total)
    return {"out": out, "sum": total}


_RUN = {
    "stream": _run_stream,
    "utterance": lambda s: s.decoder.from_indices(s.codes),
    "hifigan": lambda s: s.vocoder(s.mel),
    "unit": _run_unit,
    "stack": lambda s: residual_stack(s.x, s.units, None, s.a, s.b, final=s.final,
                                      coef_table=s.table),
    "layer": _run_layer,
    "hift": lambda s: {"spectrum": s.stft.spectrum(s.signal), "wave": s.stft.tail(s.h)},
    "cl_unit": _run_cl_unit,
    "cl_up": lambda s: channels_last_conv_transpose1d(s.x, s.up, s.weight, s.up.bias),
    "rvq": lambda s: rvq_gather_sum(s.codes, s.tables, clamp=True),
}


# ------------------------------------------------------------------ work


def _codec_work(rows: int, frames: int) -> tuple[float, float]:
    """FLOPs of the codec's convs, and its weights, codes and waveform (the gathered codebook
    rows among them) in bytes."""
    macs, weights, length, c = frames * 512 * 1536 * 7, 512 * 1536 * 7, frames, 1536
    for stride in (8, 8, 5, 6):
        half = c // 2
        macs += length * c * half * 2 * stride
        weights += c * half * 2 * stride + 3 * half * half * 8
        length *= stride
        macs += length * 3 * half * half * 8
        c = half
    macs += length * c * 7
    return 2.0 * rows * macs, 2.0 * weights + rows * (frames * 16 * (512 * 2 + 8) + length * 4)


def work(case: dict) -> dict:
    kind = case["kind"]
    rows = case.get("rows", 0)
    if kind in ("stream", "utterance"):
        streams = case.get("streams", rows)
        flops, nbytes = _codec_work(streams, case["frames"])
        if kind == "stream":  # each stream's conv histories read and written once
            nbytes += 2 * streams * 238_000
    elif kind == "hifigan":
        length, c = case["frames"], 512
        macs, weights = length * 80 * 512 * 7, 80 * 512 * 7
        for c_in, c, k, rate in UPSAMPLERS:
            macs += length * c_in * c * k
            weights += c_in * c * k + 6 * 21 * c * c
            length *= rate
            macs += length * 6 * 21 * c * c
        macs += length * c * 7
        flops = 2.0 * rows * macs
        nbytes = 2.0 * weights + rows * (case["frames"] * 80 * 4 + length * 4)
    elif kind == "unit":
        c, n = case["channels"], rows * case["samples"]
        flops, nbytes = 2.0 * n * 8 * c * c, 2.0 * 8 * c * c + n * c * 8.0
    elif kind == "stack":
        n = rows * case["samples"]
        flops = 2.0 * n * (3 * 8 * 96 * 96 + 96 * 7)
        nbytes = n * (96 * 2 + 4.0) + 3 * 8 * 96 * 96 * (1 if case["fp8"] else 2)
    elif kind == "layer":
        m, weights = rows * case["frames"], 1024 * (3072 + 1024 + 6144 + 3072)
        flops = 2.0 * m * (weights + 2 * 1024 * 72)
        # the residual stream in and out, qkv out, the window of past keys and values read
        nbytes = 2.0 * weights + m * (1024 * 8 + 3072 * 2)
        if case["warm"]:
            nbytes += 2 * 2048.0 * (m + rows * 71)
    elif kind == "hift":
        frames = case["samples"] // 4 + 1
        nbytes = 4.0 * rows * (2 * case["samples"] + 2 * 18 * frames)
        flops = 2.0 * rows * frames * 2 * 16 * 18
    elif kind == "cl_unit":
        c, n, d = case["channels"], rows * case["samples"], case["dilation"]
        flops = 2.0 * n * 8 * c * c
        nbytes = 2.0 * (8 * c * c + c * (4 * n + 6 * d * rows))
    elif kind == "cl_up":
        c_in, c_out, k, stride = UPSAMPLERS[case["stage"]]
        size, n = DTYPES[case["dtype"]].itemsize, rows * case["samples"]
        flops = 2.0 * n * c_in * c_out * k
        nbytes = float(size) * (c_in * c_out * k + n * (c_in + stride * c_out))
    else:
        n, size = rows * case["frames"], DTYPES[case["tables"]].itemsize
        flops = 1.0 * n * case["books"] * 512
        nbytes = n * ((case["books"] + 1) * 512.0 * size
                      + case["books"] * (4 if case["codes"] == "i32" else 8))
    return {"bytes": nbytes, "flops": flops}


# ------------------------------------------------------------------ tolerance


def tolerance(case: dict):
    """About four times each path's measured distance from ``exact``: 4e-3 for whole decodes in
    bf16 (16 and more layers of roundings), 3e-3 for single bf16 blocks, 6e-4 for the float16
    unit, 4e-7 for the float32 upsampler and 2e-7 for the transforms."""
    kind = case["kind"]
    if kind in ("stream", "utterance", "hifigan"):
        return {"rel": 2e-2, "max": 0.5}
    if kind == "cl_up":
        return {"rel": {"f32": 2e-6, "f16": 2e-3, "bf16": 1e-2}[case["dtype"]]}
    if kind == "cl_unit":
        return {"rel": 2.5e-3 if case["dtype"] == "f16" else 1.5e-2}
    if kind == "hift":
        return {"rel": 1e-6, "max": 1e-4}
    if kind == "rvq":
        return {"rel": 1e-2 if case["tables"] == "bf16" else 1e-6}
    return {"rel": 1e-2}


# ------------------------------------------------------------------ exact


def _snake64(x: torch.Tensor, alpha: torch.Tensor) -> torch.Tensor:
    a = alpha.to(F64)
    return x + torch.sin(a * x) ** 2 / (a + 1e-9)


def _conv64(x: torch.Tensor, node: dict, dilation: int = 1, left: int | None = None) -> torch.Tensor:
    """x [B, L, C] through a conv of L outputs: causal, or with ``left`` zeros in front."""
    w, b = _dense(node), node["bias"].to(F64)
    k = w.shape[2]
    reach, length = (k - 1) * dilation, x.shape[1]
    left = reach if left is None else left
    x = torch.nn.functional.pad(x, (0, 0, left, reach - left))
    out = b.expand(x.shape[0] * length, -1).clone()
    for j in range(k):
        out.addmm_(x[:, j * dilation:j * dilation + length].reshape(-1, x.shape[2]),
                   w[:, :, j].t().contiguous())
    return out.view(x.shape[0], length, -1)


def _up64(x: torch.Tensor, node: dict, stride: int, first: int, count: int) -> torch.Tensor:
    """``count`` samples of x [B, L, C]'s transposed conv, from sample ``first`` on."""
    w = node["weight"].to(F64)
    k, (batch, length) = w.shape[2], x.shape[:2]
    out = torch.zeros(batch, (length - 1) * stride + k, w.shape[1], dtype=F64, device=x.device)
    flat = x.reshape(-1, x.shape[2])
    for j in range(k):
        out[:, j:j + (length - 1) * stride + 1:stride] += (flat @ w[:, :, j]).view(batch, length, -1)
    return out[:, first:first + count] + node["bias"].to(F64)


def _codec64(codes: torch.Tensor, tree: dict) -> torch.Tensor:
    books = tree["codebooks"]
    x = sum(books[k][codes[:, k]].to(F64) for k in range(books.shape[0]))
    x = _conv64(x, tree["in_conv"])
    for block in tree["blocks"]:
        x = _up64(_snake64(x, block["alpha"]), block["up"], block["stride"], 0,
                  x.shape[1] * block["stride"])
        for unit in block["units"]:
            y = _conv64(_snake64(x, unit["alpha1"]), unit["conv1"], unit["dilation"])
            x = x + _conv64(_snake64(y, unit["alpha2"]), unit["conv2"])
    x = _conv64(_snake64(x, tree["final"]["alpha"]), tree["final"]["conv"])
    return torch.tanh(x).transpose(1, 2).contiguous()


def _hifigan64(mel: torch.Tensor, tree: dict) -> torch.Tensor:
    leaky = torch.nn.functional.leaky_relu
    x = _conv64(mel.transpose(1, 2).to(F64), tree["conv_pre"], left=3)
    for stage in tree["stages"]:
        k, rate = stage["up"]["weight"].shape[2], stage["rate"]
        x = _up64(leaky(x, 0.1), stage["up"], rate, (k - rate) // 2, x.shape[1] * rate)
        total = torch.zeros_like(x)
        for block in stage["resblocks"]:
            y, reach = x, (block["kernel"] - 1) // 2
            for c1, c2, d in zip(block["convs1"], block["convs2"], block["dilations"]):
                t = _conv64(leaky(y, 0.1), c1, d, left=reach * d)
                y = y + _conv64(leaky(t, 0.1), c2, left=reach)
            total += y
        x = total / 3
    x = _conv64(leaky(x, 0.01), tree["conv_post"], left=3)
    return torch.tanh(x).transpose(1, 2).contiguous()


def _layer64(w: SimpleNamespace, case: dict) -> dict:
    rows, frames = case["rows"], case["frames"]
    h = w.h.to(F64)

    def norm(x, weight):
        return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-5) * weight.to(F64)

    qkv = (norm(h, w.norm1) @ w.qkv.to(F64).t()).view(rows, frames, 3, 16, 64)
    start = (w.positions[w.slots] if case["warm"]
             else torch.zeros(rows, dtype=torch.int64, device=DEVICE))
    position = start[:, None] + torch.arange(frames, device=DEVICE)
    angle = position.to(F64)[..., None] * w.inv_freq.to(F64)
    cos, sin = (torch.cat([f(angle)] * 2, dim=-1)[:, :, None, None] for f in (torch.cos, torch.sin))
    qk = qkv[:, :, :2]
    qk = qk * cos + torch.cat([-qk[..., 32:], qk[..., :32]], dim=-1) * sin
    qkv = torch.cat([qk, qkv[:, :, 2:]], dim=2)
    out = {"qkv": qkv.reshape(rows * frames, 3072)}
    keys, values = qkv[:, :, 1], qkv[:, :, 2]
    key_position = position
    if case["warm"]:
        ring = w.slots[:, None] * w.ring
        out["keys"], out["values"] = w.keys.to(F64), w.values.to(F64)
        past = start[:, None] - 71 + torch.arange(71, device=DEVICE)
        new_rows, past_rows = (ring + p % w.ring for p in (position, past))
        keys, values = (torch.cat([out[n][past_rows].view(rows, 71, 16, 64), t], dim=1)
                        for n, t in (("keys", keys), ("values", values)))
        key_position = torch.cat([past, position], dim=1)
        out["keys"][new_rows] = qkv[:, :, 1].reshape(rows, frames, 1024)
        out["values"][new_rows] = qkv[:, :, 2].reshape(rows, frames, 1024)
    behind = position[:, :, None] - key_position[:, None]
    q, keys, values = (t.transpose(1, 2).contiguous() for t in (qkv[:, :, 0], keys, values))
    scores = (q @ keys.transpose(2, 3).contiguous()) * 0.125
    scores = scores.masked_fill(((behind < 0) | (behind >= 72))[:, None], -math.inf)
    attn = (torch.softmax(scores, dim=-1) @ values).transpose(1, 2).reshape(rows * frames, 1024)
    h = h + w.scale1.to(F64) * (attn @ w.o.to(F64).t())
    gate, up = (norm(h, w.norm2) @ w.gate_up.to(F64).t()).chunk(2, dim=-1)
    out["h"] = h + w.scale2.to(F64) * ((gate * torch.sigmoid(gate) * up) @ w.down.to(F64).t())
    return out


def _hift64(signal: torch.Tensor, h: torch.Tensor) -> dict:
    window = torch.hann_window(16, periodic=True, dtype=F64, device=DEVICE)
    spec = torch.stft(signal.to(F64), 16, 4, 16, window, center=True, pad_mode="reflect",
                      return_complex=True)
    magnitude = torch.exp(h[..., :9].to(F64)).clamp(max=100.0)
    phase = torch.sin(h[..., 9:].to(F64))
    wave = torch.istft(torch.polar(magnitude, phase).transpose(1, 2), 16, 4, 16, window, center=True)
    return {"spectrum": torch.cat([spec.real, spec.imag], dim=1), "wave": wave.clamp(-0.99, 0.99)}


def _cl_unit64(w: SimpleNamespace, case: dict) -> dict:
    def snake_beta(x, alpha, beta):
        return x + torch.sin(torch.exp(alpha.to(F64)) * x) ** 2 / (torch.exp(beta.to(F64)) + 1e-9)

    y = _conv64(w.u.to(F64), w.conv1, case["dilation"])[:, 6 * case["dilation"]:]
    total = _conv64(snake_beta(y, w.alpha1, w.beta1), w.conv2) + w.x.to(F64)
    return {"out": snake_beta(total, w.alpha2, w.beta2), "sum": total}


def exact(case: dict, seed: int):
    r, kind = _Random(seed), case["kind"]
    if kind in ("stream", "utterance"):
        tree = _codec_weights(r)
        if kind == "utterance":
            codes = r.integers(2048, case["rows"], 16, case["frames"])
            return torch.cat([_codec64(c, tree) for c in codes.split(1)])
        wave = torch.cat([_codec64(c, tree) for c in _stream_codes(r, case).split(8)])
        # the histories are the convs' own operands, in the decoder's layout
        return {"wave": wave[..., wave.shape[2] // 2:].contiguous(), "parity": None,
                "histories": None}
    if kind == "hifigan":
        tree = _hifigan_weights(r)
        mel = r.normal(case["rows"], 80, case["frames"], std=2.0) - 5.0
        return torch.cat([_hifigan64(m, tree) for m in mel.split(4)])
    if kind == "unit":
        w = _unit_weights(r, case)
        out, total = [], []
        for x in w.x.to(F64).split(1):
            y = _conv64(_snake64(x, w.alpha1), w.conv1, case["dilation"])
            total.append(x + _conv64(_snake64(y, w.alpha2), w.conv2))
            out.append(_snake64(total[-1], w.alpha3))
        return {"out": torch.cat(out), "sum": torch.cat(total)}
    if kind == "stack":
        w, waves = _stack_weights(r, case), []
        for x in w.x.split(1):
            x = x.to(F64)
            for u in w.units:
                y = _conv64(_snake64(x, u.alpha1), u.conv1, u.dilation)
                x = x + _conv64(_snake64(y, u.alpha2), u.conv2)
            waves.append(torch.tanh(_conv64(_snake64(x, w.alpha), w.final)).transpose(1, 2))
        return torch.cat(waves)
    if kind == "layer":
        return _layer64(_layer_weights(r, case), case)
    if kind == "hift":
        return _hift64(*_hift_inputs(r, case))
    if kind == "cl_unit":
        return _cl_unit64(_cl_unit_weights(r, case), case)
    if kind == "cl_up":
        w = _cl_up_weights(r, case)
        k, length = w.up["weight"].shape[2], w.x.shape[1]
        return _up64(w.x.to(F64), w.up, w.stride, w.padding,
                     (length - 1) * w.stride + k - 2 * w.padding)
    codes, tables = _rvq_inputs(r, case)
    return sum(tables[k][codes[:, k].long()].to(F64) for k in range(tables.shape[0]))
