"""``omni_bias_snake_beta``, eight channels per thread against one: the same bits. A call whose
tensors start 16 bytes in takes the eight-wide kernel, the same call on copies that start 2 bytes
further the one-wide (channel counts that are no multiple of 8 too); with and without bias,
residual and sum, float16 and bfloat16, parameters in the data type or float32, rows spaced apart,
infinities, NaN and the types' extremes among the inputs."""

from __future__ import annotations

import pytest
import torch

from sglang_omni_amd.kernels.bias_snake_beta import SnakeBetaCoefficients, fused_bias_snake_beta

pytestmark = pytest.mark.gpu


def _shifted(t: torch.Tensor) -> torch.Tensor:
    """A copy whose data starts one element past a 16-byte boundary, with t's strides."""
    size = sum((n - 1) * s for n, s in zip(t.shape, t.stride())) + 1
    buf = torch.empty(size + 1, dtype=t.dtype, device=t.device)[1:]
    out = buf.as_strided(t.shape, t.stride())
    out.copy_(t)
    return out


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("params", ["same", "float32"])
@pytest.mark.parametrize("batch,length,channels", [(1, 1, 8), (3, 37, 24), (2, 300, 192), (1, 5, 8),
                                                   (4, 1031, 96), (2, 33, 20)])
def test_eight_wide_equals_one_wide(gpu, dtype, params, batch, length, channels):
    g = torch.Generator().manual_seed(channels + length)
    pdt = dtype if params == "same" else torch.float32

    def draw(*shape, spread=3.0):
        return torch.randn(*shape, generator=g) * spread

    rows = draw(batch, length + 5, channels)
    special = torch.tensor([float("inf"), -float("inf"), float("nan"), 0.0, -0.0, 65504.0, 6e-8, 1e4])
    rows.view(-1)[: special.numel()] = special
    conv = rows.to(dtype).to(gpu)[:, :length]  # rows spaced apart
    residual = draw(batch, length, channels).to(dtype).to(gpu)
    bias = draw(channels).to(pdt).to(gpu)
    co = [draw(channels, spread=1.0).abs().to(pdt).to(gpu) for _ in range(2)]
    for has_bias in (True, False):
        for has_sum in (True, False):
            results = []
            for shift in (lambda t: t, _shifted):
                out = shift(torch.zeros_like(rows.to(dtype).to(gpu)))[:, :length]
                total = shift(torch.zeros_like(residual)) if has_sum else None
                fused_bias_snake_beta(shift(conv), bias if has_bias else None,
                                      SnakeBetaCoefficients(alpha_scale=co[0], inverse_beta=co[1]), out,
                                      residual=shift(residual) if has_sum else None, sum_out=total)
                results.append([out.contiguous()] + ([total.contiguous()] if has_sum else []))
            for a, b in zip(*results):
                assert torch.equal(a.view(torch.int16), b.view(torch.int16))
