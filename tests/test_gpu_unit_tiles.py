"""The 192-channel fused unit's LDS-DMA tiles (64, 128 and 192 positions, chosen by rounds of one
workgroup per CU): the bits of the register-staged fused form at sizes on both sides of each
choice and of each tile's edge, over one and many rows, dilations 1 to 9 and float16 / float32
streams; streamed from slot histories, whose new samples are the same; and the choice itself."""

from __future__ import annotations

import math

import pytest
import torch

from sglang_omni_amd import _native as N
from sglang_omni_amd.kernels.conv import fused_conv, pack_conv1d, plan_shapes

pytestmark = pytest.mark.gpu

C = 192
PLAN = dict(c_in=C, n_cols=C, c_out=C, taps=7, fused_unit=True)


def _unit(d, gpu):
    g = torch.Generator().manual_seed(d)
    def conv(taps, dilation):
        return pack_conv1d(torch.randn(C, C, taps, generator=g) / math.sqrt(C * taps),
                           torch.randn(C, generator=g) * 0.1, dilation=dilation).to(gpu)
    a = (torch.rand(C, generator=g) + 0.5).to(gpu)
    return conv(7, d), conv(1, 1), a


def _run(x, unit, residual, config, **kw):
    c1, c2, a = unit
    out = torch.full(x.shape, float("nan"), dtype=torch.bfloat16, device=x.device)
    total = torch.full(x.shape, float("nan"), dtype=residual.dtype, device=x.device)
    fused_conv(x, c1, out, second=c2, mid_activation=N.ACT_SNAKE, mid_a=a, mid_b=1 / a,
               residual=residual, sum_out=total, activation=N.ACT_SNAKE, act_a=1 / a, act_b=a,
               kernel=N.CONV_KERNEL_FUSED_UNIT, config=config, **kw)
    assert not out.isnan().any()
    return out, total


def _tensors(batch, length, dtype, gpu):
    g = torch.Generator().manual_seed(batch * 7 + length)
    return (torch.randn(batch, length, C, generator=g).to(torch.bfloat16).to(gpu),
            torch.randn(batch, length, C, generator=g).to(dtype).to(gpu))


@pytest.mark.parametrize("batch,length,tile", [
    (1, 1, 64), (1, 63, 64), (1, 65, 64), (3, 191, 64), (2, 64, 64), (1, 16384, 64), (1, 16385, 128),
    (5, 5003, 128), (8, 4096, 128), (7, 4800, 192), (1, 49152, 192), (12, 5003, 128), (1, 65537, 192)])
def test_tiles_give_the_staged_forms_bits(gpu, batch, length, tile):
    plan = plan_shapes(batch=batch, length=length, dilation=9, kernel=N.CONV_KERNEL_FUSED_UNIT,
                       config=1, **PLAN)
    assert plan.workgroups == -(-batch * length // tile)
    for d, dtype in ((9, torch.float16), (1, torch.float32), (3, torch.float16)):
        unit = _unit(d, gpu)
        x, residual = _tensors(batch, length, dtype, gpu)
        for got, want in zip(_run(x, unit, residual, 1), _run(x, unit, residual, 2)):
            assert torch.equal(got, want), d


@pytest.mark.parametrize("batch,length", [(3, 200), (9, 2000), (9, 4000), (1, 20)])
@pytest.mark.parametrize("cold", [False, True])
def test_streamed_history(gpu, batch, length, cold):
    unit = _unit(9, gpu)
    x, residual = _tensors(batch, length, torch.float16, gpu)
    slots, h = batch + 2, unit[0].left_pad
    g = torch.Generator().manual_seed(3)
    pool = torch.randn(slots, 2, h, C, generator=g).to(torch.bfloat16).to(gpu)
    slot_index = torch.randperm(slots, generator=g)[:batch].to(gpu)
    slot_index[-1] = -1
    results = []
    for config in (1, 2):
        history = pool.clone()
        results.append((*_run(x, unit, residual, config, history=history, history_cold=cold,
                              slot_index=slot_index,
                              slot_parity=torch.arange(slots, device=gpu)), history))
    for got, want in zip(*results):
        assert torch.equal(got, want)
