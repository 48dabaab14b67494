"""``omni_gemm`` / ``omni_gemm_rope_kv`` at few rows: the automatic choice's tiles with K in stages
of 256 and 128 (16 x 32, 32 x 32, 32 x 64; 16, 32, 64 x 64 with the rotary epilogue) add every
element's products in the order of the forced tiles, so their results are the same bits. Row counts
at the tiles' edges and on both sides of each choice's line on 256 compute units; K of one stage,
fewer stages than the ring, odd multiples, and K that only the stages of 64 divide."""

from __future__ import annotations

import math

import pytest
import torch

from sglang_omni_amd.kernels.gemm import (GELU, SCALED_RESIDUAL, SILU_MUL, STORE, linear,
                                          linear_rope_kv, pack_linear)

pytestmark = pytest.mark.gpu


def _operands(gpu, rows, k, n, seed, gated=False):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(rows, k, generator=g).to(torch.bfloat16).to(gpu)
    w = torch.randn(n, k, generator=g) / math.sqrt(k)
    return x, pack_linear(w, torch.randn(n, generator=g) * 0.1, gated=gated).to(gpu)


@pytest.mark.parametrize("epilogue", [STORE, SILU_MUL, GELU, SCALED_RESIDUAL])
@pytest.mark.parametrize("k,n", [(256, 64), (512, 1024), (1024, 1024), (3072, 1024), (1024, 4096),
                                 (768, 320), (640, 1024), (192, 1024)])
def test_same_bits_as_the_forced_tiles(gpu, epilogue, k, n):
    x, lw = _operands(gpu, 520, k, n, k + n, gated=epilogue == SILU_MUL)
    cols = lw.out_features
    g = torch.Generator().manual_seed(1)
    residual = torch.randn(520, cols, generator=g).to(gpu)
    scale = torch.rand(cols, generator=g).to(gpu)

    def run(rows, config):
        scaled = epilogue == SCALED_RESIDUAL
        out = torch.full((rows + 1, cols), float("nan"), device=gpu,
                         dtype=torch.float32 if scaled else torch.bfloat16)
        kw = {"scale": scale, "residual": residual[:rows]} if scaled else {}
        linear(x[:rows], lw, out[:rows], epilogue=epilogue, config=config, **kw)
        assert out[rows].isnan().all()  # nothing past the last row
        return out[:rows]

    whole = run(520, 2)
    for rows in (1, 15, 16, 17, 33, 64, 80, 128, 129, 255, 257, 500, 520):
        assert torch.equal(run(rows, 0), whole[:rows]), rows


@pytest.mark.parametrize("k", [256, 512, 1024, 1280, 192])
@pytest.mark.parametrize("heads,kv_heads", [(16, 16), (4, 2)])
def test_rope_same_bits_as_the_forced_tile(gpu, k, heads, kv_heads):
    n = (heads + 2 * kv_heads) * 64
    ring_frames = 9
    inv = (1.0 / (10000.0 ** (torch.arange(0, 64, 2, dtype=torch.float32) / 64))).to(gpu)
    for batch, frames in ((1, 1), (5, 3), (16, 5), (17, 5), (33, 5), (34, 5), (11, 31), (70, 5)):
        x, lw = _operands(gpu, batch * frames, k, n, batch)
        positions = torch.arange(batch, device=gpu) * 37
        slots = torch.arange(batch - 1, -1, -1, device=gpu)

        def run(config):
            qkv = torch.full((batch * frames + 1, n), float("nan"), dtype=torch.bfloat16, device=gpu)
            rings = [torch.zeros(batch * ring_frames, kv_heads * 64, dtype=torch.bfloat16, device=gpu)
                     for _ in range(2)]
            if frames > ring_frames:  # a first decode longer than the ring has none
                linear_rope_kv(x, lw, qkv[:-1], batch, heads, kv_heads, 64, inv, config=config)
            else:
                linear_rope_kv(x, lw, qkv[:-1], batch, heads, kv_heads, 64, inv, cold=False,
                               slot_index=slots, positions=positions, key_ring=rings[0],
                               value_ring=rings[1], ring_frames=ring_frames, config=config)
            assert qkv[-1].isnan().all()
            return [qkv[:-1], *rings]

        for got, want in zip(run(0), run(1)):
            assert torch.equal(got, want), (batch, frames)
