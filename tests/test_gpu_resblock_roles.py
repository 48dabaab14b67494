"""``omni_resblock_pair`` at the edges of its tiles (256 - (k - 1) output positions, workgroups that
take several tiles, rows of a few positions) and over the forms its epilogue takes (no bias, no
residual, float32 output, Snake / tanh activation, strided tensors, float16 and float32 streams,
the mix with and without the stream): the bits of the two ``omni_conv1d_fused`` launches, and
nothing written between or past the rows."""

from __future__ import annotations

import math

import pytest
import torch

from sglang_omni_amd import _native as N
from sglang_omni_amd.kernels.conv import fused_conv, pack_conv1d, resblock_pair

pytestmark = pytest.mark.gpu

SLOPE = 0.1


def _pair(k, d, gpu, bias=True):
    g = torch.Generator().manual_seed(100 * k + d)
    def conv(dilation):
        return pack_conv1d(torch.randn(32, 32, k, generator=g) / math.sqrt(32 * k),
                           torch.randn(32, generator=g) * 0.1 if bias else None,
                           dilation=dilation, causal=False).to(gpu)
    return conv(d), conv(1)


def _rows(batch, length, pitch, dtype, gpu, seed=None):
    """[batch, length, 32], the last of each of a NaN buffer's rows of `pitch` elements (or random)."""
    buf = torch.full((batch, length + 3, pitch), float("nan"), dtype=dtype, device=gpu)
    view = buf[:, :length, pitch - 32:]
    if seed is not None:
        g = torch.Generator().manual_seed(seed)
        view.copy_(torch.randn(batch, length, 32, generator=g).to(dtype))
    return buf, view


def _both(x, c1, c2, gpu, *, out_dtype=torch.bfloat16, stream=torch.float16, pitch=32,
          residual=True, mix=False, sum_out=True, out=True, **kw):
    batch, length, _ = x.shape
    if residual:
        kw["residual"] = _rows(batch, length, pitch, stream, gpu, 7)[1]
    if mix:
        kw["mix"] = (_rows(batch, length, pitch, stream, gpu, 8)[1],
                     _rows(batch, length, pitch, stream, gpu, 9)[1], 1.0 / 3.0)
    results = []
    for paired in (False, True):
        buffers = []
        o = s = None
        if out:
            buf, o = _rows(batch, length, pitch, out_dtype, gpu)
            buffers.append(buf)
        if sum_out:
            buf, s = _rows(batch, length, pitch, stream, gpu)
            buffers.append(buf)
        if paired:
            resblock_pair(x, c1, c2, o, slope1=SLOPE, sum_out=s, **kw)
        else:
            h = torch.empty(batch, length, 32, dtype=torch.bfloat16, device=gpu)
            fused_conv(x, c1, h, activation=N.ACT_LEAKY_RELU, slope=SLOPE)
            fused_conv(h, c2, o, sum_out=s, **kw)
        results.append(buffers)
    for want, got in zip(*results):
        assert not want[:, :length, want.shape[2] - 32:].isnan().any()
        bits = torch.int32 if want.dtype == torch.float32 else torch.int16
        assert torch.equal(got.view(bits), want.view(bits))  # the NaNs around the rows too


@pytest.mark.parametrize("k", [3, 7, 11])
@pytest.mark.parametrize("d", [1, 2, 5])
def test_tile_edges(gpu, k, d):
    c1, c2 = _pair(k, d, gpu)
    bp = 256 - (k - 1)
    for batch, length in ((1, 1), (2, 3), (3, bp - 1), (1, bp), (2, bp + 1), (1, 2 * bp + 17),
                          (2, 1100 * bp + 5), (700, 40)):
        x = _rows(batch, length, 32, torch.bfloat16, gpu, 5)[1]
        _both(x, c1, c2, gpu, activation=N.ACT_LEAKY_RELU, slope=SLOPE)


@pytest.mark.parametrize("k", [3, 7, 11])
@pytest.mark.parametrize("stream", [torch.float16, torch.float32])
def test_epilogue_forms(gpu, k, stream):
    c1, c2 = _pair(k, 3, gpu)
    plain1, plain2 = _pair(k, 3, gpu, bias=False)
    a = torch.rand(32, device=gpu) + 0.5
    x = _rows(2, 777, 48, torch.bfloat16, gpu, 6)[1]  # strided rows
    lrelu = dict(activation=N.ACT_LEAKY_RELU, slope=0.01)
    for pitch in (32, 40, 36):  # (36: rows and a first element 8 bytes past a 16-byte boundary)
        kw = dict(stream=stream, pitch=pitch)
        _both(x, plain1, plain2, gpu, residual=False, sum_out=False, **kw)
        _both(x, c1, c2, gpu, residual=False, **kw, **lrelu)
        _both(x, c1, c2, gpu, out=False, **kw)
        _both(x, c1, c2, gpu, mix=True, sum_out=False, **kw, **lrelu)
        _both(x, c1, c2, gpu, mix=True, **kw)
        _both(x, c1, c2, gpu, out_dtype=torch.float32, activation=N.ACT_TANH, **kw)
        _both(x, c1, c2, gpu, activation=N.ACT_SNAKE, act_a=a, act_b=1 / a, **kw)


def test_the_float32_mix_at_three_taps_moves_its_bytes_as_fast_as_the_float16_mix(gpu):
    """512 bytes a position against 320. With registers spilled to memory it took 2.1 times the float16
    mix's time instead of 1.6 (each the least of ten runs at 1.3 M positions)."""
    c1, c2 = _pair(3, 5, gpu)
    x = torch.randn(4, 325366, 32, device=gpu).to(torch.bfloat16)
    best = {}
    for stream in (torch.float16, torch.float32):
        residual, a, b = (torch.randn(4, 325366, 32, device=gpu).to(stream) for _ in range(3))
        out = torch.empty_like(x)
        best[stream] = float("inf")
        for _ in range(12):
            start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            start.record()
            for _ in range(5):
                resblock_pair(x, c1, c2, out, slope1=SLOPE, residual=residual, mix=(a, b, 1.0 / 3.0),
                              activation=N.ACT_LEAKY_RELU, slope=SLOPE)
            end.record()
            torch.cuda.synchronize()
            best[stream] = min(best[stream], start.elapsed_time(end))
    assert best[torch.float32] <= 1.85 * best[torch.float16], best
