"""The smaller LDS-DMA tiles (``CONV_KERNEL_DMA_MID``): each entry gives the bits of the large tiles
on shapes at its edges (positions around 64, 128 and 256, several rows per tile, rows split across
tiles, a column tile with columns past the end), with the residual / float16 stream epilogue and
from slot histories, whose new samples it writes alike; and the automatic choice takes each entry
and its neighbours without a change of bits. The large tiles are held against float64 in
``test_gpu_tiles``."""

from __future__ import annotations

import math

import pytest
import torch

from sglang_omni_amd import _native as N
from sglang_omni_amd.kernels.conv import (fused_conv, pack_conv1d, pack_conv_transpose1d,
                                          plan_shapes)

pytestmark = pytest.mark.gpu

ENTRIES = 3


def _conv(taps, c_in, c_out, d, gpu):
    g = torch.Generator().manual_seed(taps * 1000 + c_in + c_out)
    if taps == 2:
        return pack_conv_transpose1d(torch.randn(c_in, c_out, 8, generator=g) / math.sqrt(2 * c_in),
                                     torch.randn(c_out, generator=g) * 0.1, stride=4).to(gpu)
    return pack_conv1d(torch.randn(c_out, c_in, taps, generator=g) / math.sqrt(c_in * taps),
                       torch.randn(c_out, generator=g) * 0.1, dilation=d).to(gpu)


def _run(x, conv, kernel, config, residual, a, **kw):
    shape = (x.shape[0], x.shape[1], conv.n_cols)
    out = torch.full(shape, float("nan"), dtype=torch.bfloat16, device=x.device)
    total = torch.full(shape, float("nan"), dtype=torch.float16, device=x.device)
    if conv.taps == 1:
        kw["residual"] = residual
    fused_conv(x, conv, out, kernel=kernel, config=config, sum_out=total, activation=N.ACT_SNAKE,
               act_a=a, act_b=1 / a, **kw)
    assert not out.isnan().any() and not total.isnan().any()
    return out, total


def _reference(x, conv, residual, a, **kw):
    for config in (4, 3, 2, 1):  # a large tile that fits
        try:
            return _run(x, conv, N.CONV_KERNEL_DMA, config, residual, a, **kw)
        except N.OmniCodecError as e:
            if e.status != N.UNSUPPORTED:
                raise
    return None


@pytest.mark.parametrize("taps,c_in,c_out,d", [(7, 384, 384, 9), (7, 96, 256, 1), (7, 192, 192, 3),
                                               (1, 384, 384, 1), (1, 768, 192, 1),
                                               (2, 768, 96, 1), (2, 448, 64, 1)])
def test_entries_give_the_large_tiles_bits(gpu, taps, c_in, c_out, d):
    conv = _conv(taps, c_in, c_out, d, gpu)
    a = torch.rand(conv.c_out, device=gpu) + 0.5
    ran = {k: 0 for k in range(1, ENTRIES + 1)}
    for batch, length in ((1, 1), (1, 63), (1, 64), (1, 129), (1, 255), (1, 257), (3, 100), (2, 700),
                          (5, 31)):
        g = torch.Generator().manual_seed(length)
        x = torch.randn(batch, length, c_in, generator=g).to(torch.bfloat16).to(gpu)
        res = torch.randn(batch, length, conv.n_cols, generator=g).half().to(gpu)
        want = _reference(x, conv, res, a)
        for config in ran:
            try:
                got = _run(x, conv, N.CONV_KERNEL_DMA_MID, config, res, a)
            except N.OmniCodecError as e:
                assert e.status == N.UNSUPPORTED
                continue
            ran[config] += 1
            if want is not None:
                assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]), (batch, length)
        if want is not None:
            auto = _run(x, conv, N.CONV_KERNEL_AUTO, 0, res, a)
            assert torch.equal(auto[0], want[0]) and torch.equal(auto[1], want[1])
    # (an entry may not serve a layer: its stages take 1 to 4 chunks)
    assert sum(n >= 3 for n in ran.values()) >= 1, ran


@pytest.mark.parametrize("taps,d", [(7, 9), (2, 1)])
def test_streamed_history(gpu, taps, d):
    conv = _conv(taps, 384, 384 if taps == 7 else 96, d, gpu)
    a = torch.rand(conv.c_out, device=gpu) + 0.5
    batch, length, slots, h = 3, 300, 5, conv.left_pad
    g = torch.Generator().manual_seed(2)
    x = torch.randn(batch, length, 384, generator=g).to(torch.bfloat16).to(gpu)
    pool = torch.randn(slots, 2, h, 384, generator=g).to(torch.bfloat16).to(gpu)
    kw = dict(slot_index=torch.tensor([4, -1, 1], device=gpu),
              slot_parity=torch.tensor([0, 0, 0, 0, 1], device=gpu))

    def run(kernel, config, cold):
        history = pool.clone()
        return (*_run(x, conv, kernel, config, None, a, history=history, history_cold=cold, **kw),
                history)

    for cold in (False, True):
        want = run(N.CONV_KERNEL_DMA, 3, cold)
        for config in range(1, ENTRIES + 1):
            for got, ref in zip(run(N.CONV_KERNEL_DMA_MID, config, cold), want):
                assert torch.equal(got, ref), (cold, config)


def test_automatic_choice_and_refusals():
    """The decoder's layers for an utterance of 250 frames take the smaller tiles, a loaded step
    the large ones; E4M3 weights and activated operands have no smaller tiles; what the large
    tiles refuse stays refused."""
    layers = [(768, 768, 768, 7, 9, 2000), (768, 768, 768, 1, 1, 2000), (384, 384, 384, 7, 9, 16000),
              (384, 384, 384, 1, 1, 16000), (1536, 6144, 768, 2, 1, 250), (768, 3072, 384, 2, 1, 2000)]
    for c_in, n_cols, c_out, taps, d, positions in layers:
        kw = dict(c_in=c_in, n_cols=n_cols, c_out=c_out, taps=taps, dilation=d,
                  left_pad=1 if taps == 2 else None)
        plan = plan_shapes(batch=1, length=positions, **kw)
        assert plan.kernel == N.CONV_KERNEL_DMA_MID and plan.configs == ENTRIES
        assert plan_shapes(batch=1, length=positions, fp8=True, **kw).kernel == N.CONV_KERNEL_DMA
        for bad in (dict(fp8=True), dict(in_activation=N.ACT_SNAKE)):
            with pytest.raises(N.OmniCodecError, match="status 2"):
                plan_shapes(batch=1, length=positions, kernel=N.CONV_KERNEL_DMA_MID, config=1,
                            **kw, **bad)
    with pytest.raises(N.OmniCodecError, match="status 2"):
        plan_shapes(batch=64, length=2, c_in=384, n_cols=384, c_out=384, taps=7, dilation=9)
