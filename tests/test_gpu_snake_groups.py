"""``omni_bias_snake_beta``, eight channels per thread against one: the same bits. A call of 2^19
elements and more whose tensors start 16 bytes in takes the eight-wide kernel, the same call on
copies that start 2 bytes further the one-wide (fewer elements and channel counts that are no
multiple of 8 too); with and without bias,
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
                                                   (4, 1031, 96), (2, 33, 20),
                                                   # 2^19 elements and more: eight-wide
                                                   (1, 65536, 8), (1, 65535, 8), (3, 7001, 32),
                                                   (2, 1500, 192), (17, 33, 1000), (2, 26301, 20)])
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


def test_a_small_call_takes_no_longer_than_an_unaligned_one(gpu):
    """Eight channels per thread took 3.2 us where one takes 2.4 (20 000 elements); the unaligned copy
    always runs one-wide. Each the least of ten replays of 20 calls; 15 % for the clock."""
    x = torch.randn(1, 208, 96, device=gpu, dtype=torch.float16)
    co = SnakeBetaCoefficients(alpha_scale=torch.rand(96, device=gpu, dtype=torch.float16),
                               inverse_beta=torch.rand(96, device=gpu, dtype=torch.float16))
    graphs = []
    side = torch.cuda.Stream()
    for t in (x, _shifted(x)):
        out = torch.empty_like(x)
        with torch.cuda.stream(side):
            fused_bias_snake_beta(t, None, co, out)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            for _ in range(20):
                fused_bias_snake_beta(t, None, co, out)
        graphs.append((graph, out))
    start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    best = [float("inf")] * 2
    for _ in range(10):
        for i, (graph, _) in enumerate(graphs):
            start.record()
            graph.replay()
            end.record()
            torch.cuda.synchronize()
            best[i] = min(best[i], start.elapsed_time(end))
    assert best[0] <= 1.15 * best[1]
