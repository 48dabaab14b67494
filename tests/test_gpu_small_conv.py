"""The small-call conv kernels (``CONV_KERNEL_SMALL``): every configuration on shapes at its edges
gives the bits of the LDS-DMA tiles, alone, with every epilogue, from slot histories and in K
slices; and the residual unit those of the fused form. One product order for both, so equality is
exact; the LDS-DMA tiles themselves are held against float64 in ``test_gpu_tiles``."""

from __future__ import annotations

import pytest
import torch

from sglang_omni_amd import _native as N
from sglang_omni_amd.kernels.conv import (
    fused_conv,
    pack_conv1d,
    pack_conv_transpose1d,
    plan_shapes,
    splitk_conv,
)

pytestmark = pytest.mark.gpu

CONFIGS = 9
# (taps, c_in, c_out, dilation, rows, positions): one row below a tile, rows across tiles, many
# short rows (a halo per row), several slabs (768 and 1536 channels), the last group partial
SHAPES = [(7, 768, 768, 9, 1, 32), (7, 768, 192, 1, 3, 50), (7, 192, 192, 9, 2, 130),
          (7, 96, 64, 3, 5, 7), (7, 512, 96, 1, 1, 4), (7, 224, 48, 1, 1, 100),
          (1, 768, 192, 1, 1, 33), (1, 192, 192, 1, 3, 100), (1, 96, 16, 1, 1, 1),
          (2, 1536, 96, 1, 1, 5), (2, 384, 32, 1, 9, 3), (2, 96, 80, 1, 2, 65)]


def bits(gpu, shape, seed, dtype=torch.bfloat16, std=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=g) * std).to(dtype).to(gpu)


def packed_conv(gpu, taps, c_in, c_out, dilation):
    w = bits("cpu", (c_out, c_in, taps), 1, torch.float32, (c_in * taps) ** -0.5)
    b = bits("cpu", (c_out,), 2, torch.float32)
    if taps == 2:  # the polyphase form of a transposed conv of stride 3
        wt = bits("cpu", (c_in, c_out, 6), 1, torch.float32, (c_in * 2) ** -0.5)
        return pack_conv_transpose1d(wt, b, stride=3).to(gpu)
    return pack_conv1d(w, b, dilation=dilation).to(gpu)


def forced(kernel, config, x, conv, out, **kw):
    """fused_conv on a named entry; False where it does not take the call."""
    try:
        fused_conv(x, conv, out, kernel=kernel, config=config, **kw)
    except N.OmniCodecError as err:
        assert err.status == N.UNSUPPORTED
        return False
    return True


def reference(x, conv, out, **kw):
    """The LDS-DMA tile's result: its list's first entry that fits."""
    assert any(forced(N.CONV_KERNEL_DMA, c, x, conv, out, **kw) for c in range(1, 5)) or \
        forced(N.CONV_KERNEL_STAGED, 9, x, conv, out, **kw)


@pytest.mark.parametrize("taps,c_in,c_out,dilation,rows,positions", SHAPES)
def test_every_configuration_gives_the_large_tiles_bits(gpu, taps, c_in, c_out, dilation, rows,
                                                        positions):
    conv = packed_conv(gpu, taps, c_in, c_out, dilation)
    n = conv.n_cols
    x = bits(gpu, (rows, positions, c_in), 3)
    a, b = bits(gpu, (c_out,), 4, torch.float32).exp(), bits(gpu, (c_out,), 5, torch.float32)
    ran = 0
    for rdt in (torch.float16, torch.float32):
        res, m1, m2 = (bits(gpu, (rows, positions, n), s, rdt) for s in (6, 7, 8))
        cases = [(torch.bfloat16, {}),
                 (torch.bfloat16, dict(residual=res, activation=N.ACT_SNAKE, act_a=a, act_b=b)),
                 (torch.float32, dict(residual=res, mix=(m1, m2, 1 / 3), slope=0.1,
                                      activation=N.ACT_LEAKY_RELU))]
        for odt, kw in cases:
            sums = [torch.empty_like(res), torch.zeros_like(res)] if "residual" in kw else [None] * 2
            want = torch.empty(rows, positions, n, dtype=odt, device=gpu)
            reference(x, conv, want, sum_out=sums[0], **kw)
            for config in range(1, CONFIGS + 1):
                got = torch.zeros_like(want)
                if not forced(N.CONV_KERNEL_SMALL, config, x, conv, got, sum_out=sums[1], **kw):
                    continue
                ran += 1
                assert torch.equal(got, want), (config, odt)
                assert sums[0] is None or torch.equal(sums[1], sums[0])
    assert ran >= 6


@pytest.mark.parametrize("taps,c_in,c_out,dilation", [(7, 768, 192, 9), (7, 192, 192, 3),
                                                      (2, 1536, 96, 1)])
@pytest.mark.parametrize("cold", [True, False])
def test_slot_histories_are_read_and_written_alike(gpu, taps, c_in, c_out, dilation, cold):
    """Rows on shuffled slots of mixed parity, one row outside the pool, chunks shorter and longer
    than the history: outputs and both copies of every slot."""
    conv = packed_conv(gpu, taps, c_in, c_out, dilation)
    h = conv.left_pad
    for rows, positions in ((3, 5), (1, 80)):
        x = bits(gpu, (rows, positions, c_in), 3)
        index = torch.tensor([4, 0, 9][:rows], device=gpu)
        parity = torch.tensor([0, 1, 0, 1, 3], device=gpu)
        pool = bits(gpu, (5, 2, h, c_in), 9)
        results = []
        for kernel in (N.CONV_KERNEL_DMA, N.CONV_KERNEL_SMALL):
            for config in range(1, CONFIGS + 1):
                hist = pool.clone()
                out = torch.zeros(rows, positions, conv.n_cols, dtype=torch.bfloat16, device=gpu)
                if kernel == N.CONV_KERNEL_DMA and config > 4:
                    continue
                if forced(kernel, config, x, conv, out, history=hist, slot_index=index,
                          slot_parity=parity, history_cold=cold):
                    results.append((kernel, config, out, hist))
        assert results[0][0] == N.CONV_KERNEL_DMA and results[-1][0] == N.CONV_KERNEL_SMALL
        for kernel, config, out, hist in results[1:]:
            assert torch.equal(out, results[0][2]), (kernel, config)
            assert torch.equal(hist, results[0][3]), (kernel, config)


@pytest.mark.parametrize("frames", [1, 4, 20])
def test_k_slices_add_up_as_the_reduction_does(gpu, frames):
    conv = packed_conv(gpu, 7, 512, 1536, 1)
    x = bits(gpu, (2, frames, 512), 3)
    a = bits(gpu, (1536,), 4, torch.float32).exp()
    work = torch.full((4 * 2 * frames * 1536,), float("nan"), device=gpu)
    got, want = (torch.zeros(2, frames, 1536, dtype=torch.bfloat16, device=gpu) for _ in range(2))
    kw = dict(k_splits=4, workspace=work, activation=N.ACT_SNAKE, act_a=a, act_b=a)
    splitk_conv(x, conv, got, **kw)
    assert bool(work.isnan().all())  # no partials: the slices were added in registers
    splitk_conv(x, conv, want, kernel=N.CONV_KERNEL_DMA, config=1, **kw)
    assert torch.equal(got, want)


@pytest.mark.parametrize("rows,positions,dilation", [(1, 1280, 9), (3, 33, 9), (7, 20, 1), (1, 1, 3)])
@pytest.mark.parametrize("stream", [torch.float16, torch.float32])
def test_the_residual_unit_gives_the_fused_forms_bits(gpu, rows, positions, dilation, stream):
    c1, c2 = packed_conv(gpu, 7, 192, 192, dilation), packed_conv(gpu, 1, 192, 192, 1)
    x, res = bits(gpu, (rows, positions, 192), 3), bits(gpu, (rows, positions, 192), 6, stream)
    a, b = bits(gpu, (192,), 4, torch.float32).exp(), bits(gpu, (192,), 5, torch.float32)
    pool = bits(gpu, (8, 2, c1.left_pad, 192), 9)
    index, parity = torch.arange(rows, device=gpu), torch.arange(8, device=gpu)
    results = []
    for kernel, configs in ((N.CONV_KERNEL_FUSED_UNIT, (1, 2, 3)), (N.CONV_KERNEL_SMALL, (1,))):
        for config in configs:
            hist, out, total = pool.clone(), torch.zeros_like(x), torch.zeros_like(res)
            if forced(kernel, config, x, c1, out, second=c2, mid_activation=N.ACT_SNAKE, mid_a=a,
                      mid_b=b, residual=res, sum_out=total, activation=N.ACT_SNAKE, act_a=b.exp(),
                      act_b=a, history=hist, slot_index=index, slot_parity=parity):
                results.append((kernel, out, total, hist))
    assert len(results) > 1 and results[-1][0] == N.CONV_KERNEL_SMALL
    for _, *tensors in results[1:]:
        assert all(torch.equal(t, r) for t, r in zip(tensors, results[0][1:]))
