"""The conv launcher's plan and forced-configuration entry points without a GPU: the tile lists
have the lengths the forced-tile GPU tests sweep, the benchmarked workloads' layer shapes plan to
entries of those lists, and contract violations are refused before anything runs."""

from __future__ import annotations

import ctypes

import pytest

from sglang_omni_amd import _native as N
from sglang_omni_amd.kernels.conv import plan_shapes, plan_stack_shapes
from tests.test_gpu_tiles import (
    DMA_LIST,
    FUSED_LIST,
    NARROW128_DMA_LIST,
    NARROW_DMA_LIST,
    STAGED11_LIST,
    STAGED_LIST,
)


def test_list_lengths_match_the_forced_tile_sweep():
    for taps, n in DMA_LIST.items():
        c_out = 96
        n_cols = 6 * c_out if taps == 2 else c_out
        for fp8 in (False, True):  # E4M3 weights take the same tile lists
            plan = plan_shapes(batch=2, length=300, c_in=192, n_cols=n_cols, c_out=c_out,
                               taps=taps, left_pad=1 if taps == 2 else None, fp8=fp8)
            assert plan.kernel == N.CONV_KERNEL_DMA and plan.configs == n
    staged = plan_shapes(batch=2, length=300, c_in=96, n_cols=192, c_out=192, taps=7, fp8=True,
                         in_activation=N.ACT_SNAKE)
    assert staged.kernel == N.CONV_KERNEL_STAGED and staged.configs == STAGED_LIST
    s11 = plan_shapes(batch=2, length=300, c_in=64, n_cols=64, c_out=64, taps=11, dilation=5,
                      left_pad=25, in_activation=N.ACT_LEAKY_RELU)
    assert s11.kernel == N.CONV_KERNEL_STAGED11 and s11.configs == STAGED11_LIST
    for taps in NARROW_DMA_LIST:  # narrow layers with a ready bf16 operand
        for cols in (256, 128, 64, 32) if taps == 3 else (128, 64, 32):
            n = (NARROW128_DMA_LIST if cols > 64 else NARROW_DMA_LIST)[taps]
            plan = plan_shapes(batch=2, length=300, c_in=cols, n_cols=cols, c_out=cols,
                               taps=taps, dilation=5, left_pad=(taps - 1) * 5 // 2)
            assert plan.kernel == N.CONV_KERNEL_DMA and plan.configs == n
    fused = plan_shapes(batch=2, length=300, c_in=96, n_cols=96, c_out=96, taps=7, dilation=9,
                        fused_unit=True)
    assert fused.kernel == N.CONV_KERNEL_FUSED_UNIT and fused.configs == FUSED_LIST


@pytest.mark.parametrize("layer", [
    # (name, c_in, n_cols, c_out, taps, dilation, left_pad, fused) at 64 streams x 12 frames
    ("in_conv", 512, 1536, 1536, 7, 1, None, False, 12),
    ("block1.up", 768, 8 * 384, 384, 2, 1, 1, False, 96),
    ("block1.k7d9", 384, 384, 384, 7, 9, None, False, 768),
    ("block1.k1", 384, 384, 384, 1, 1, None, False, 768),
    ("block2.unit", 192, 192, 192, 7, 3, None, True, 3840),
    ("block3.up", 192, 6 * 96, 96, 2, 1, 1, False, 3840),
])
def test_streaming_step_layers_plan_to_swept_entries(layer):
    name, c_in, n_cols, c_out, taps, d, left, fused, length = layer
    plan = plan_shapes(batch=64, length=length, c_in=c_in, n_cols=n_cols, c_out=c_out, taps=taps,
                       dilation=d, left_pad=left, fused_unit=fused, history=True)
    assert 1 <= plan.config <= plan.configs
    assert plan.workgroups >= 64
    if plan.kernel == N.CONV_KERNEL_DMA:
        assert plan.configs == DMA_LIST[taps]


def test_forced_choice_contract():
    kw = dict(batch=2, length=300, c_in=192, n_cols=192, c_out=192, taps=7, dilation=3)
    # a family that cannot serve the call, and entries past the list, are "unsupported"
    with pytest.raises(N.OmniCodecError, match="status 2"):
        plan_shapes(**kw, kernel=N.CONV_KERNEL_FUSED_UNIT, config=1)
    with pytest.raises(N.OmniCodecError, match="status 2"):
        plan_shapes(**kw, kernel=N.CONV_KERNEL_DMA, config=DMA_LIST[7] + 1)
    # LDS-DMA copies the operand as it is: an operand activated on the way in never takes it
    with pytest.raises(N.OmniCodecError, match="status 2"):
        plan_shapes(**kw, in_activation=N.ACT_SNAKE, kernel=N.CONV_KERNEL_DMA, config=1)
    assert plan_shapes(**kw, fp8=True, kernel=N.CONV_KERNEL_DMA, config=1).config == 1
    # an unknown family or a configuration without a family is an invalid argument
    with pytest.raises(N.OmniCodecError, match="status 1"):
        plan_shapes(**kw, kernel=9, config=1)
    with pytest.raises(N.OmniCodecError, match="status 1"):
        plan_shapes(**kw, kernel=N.CONV_KERNEL_AUTO, config=2)
    # the forced launch refuses the automatic family, and a null argument block
    lib = N.load_library()
    assert lib.omni_conv1d_fused_with(None, N.CONV_KERNEL_DMA, 1, None) == N.INVALID_ARG
    args = N.ConvArgs()
    assert lib.omni_conv1d_fused_with(ctypes.byref(args), N.CONV_KERNEL_AUTO, 0, None) == N.INVALID_ARG


def test_an_empty_call_plans_nothing():
    plan = plan_shapes(batch=0, length=12, c_in=96, n_cols=96, c_out=96, taps=7)
    assert plan.kernel == N.CONV_KERNEL_AUTO and plan.config == 0


@pytest.mark.parametrize("channels,length", [(256, 4000), (128, 20000), (64, 60000), (32, 240000)])
@pytest.mark.parametrize("taps", [3, 7, 11])
def test_hifigan_resblock_convs_plan_to_their_tiles(channels, length, taps):
    """HiFiGAN's ResBlock convs at 16 clips x 500 mel frames ('same' padding, dilations 1 and 5)
    take the families and entries their measurements chose: LDS-DMA for all but the 256-channel
    k = 11 convs (register-staged), the one-buffer-ring entries first where c_in is one stage."""
    for d in (1, 5):
        plan = plan_shapes(batch=16, length=length, c_in=channels, n_cols=channels,
                           c_out=channels, taps=taps, dilation=d, left_pad=(taps - 1) * d // 2)
        if channels == 256 and taps == 11:
            assert plan.kernel == N.CONV_KERNEL_STAGED11
            continue
        assert plan.kernel == N.CONV_KERNEL_DMA
        if channels == 256 and taps == 7:
            assert plan.configs == DMA_LIST[7]
        elif channels >= 128:
            assert plan.configs == NARROW128_DMA_LIST[taps]
        else:
            assert plan.configs == NARROW_DMA_LIST[taps]
        # 64 channels: the two-chunk one-stage entry (k = 3) or the 64-column entry follows the
        # 32-column one-stage entry, which needs c_in = 32
        assert plan.config == (2 if channels == 64 else 1)
        assert plan.workgroups >= 256


@pytest.mark.parametrize("layer", [
    # a decoder layer at one stream of 4 frames, and at 64 streams of 12
    ("block0.k7", 768, 768, 768, 7, 9, 32), ("block0.k1", 768, 768, 768, 1, 1, 32),
    ("block0.up", 1536, 8 * 768, 768, 2, 1, 4), ("block1.k7", 384, 384, 384, 7, 3, 256),
    ("block1.up", 768, 8 * 384, 384, 2, 1, 32), ("block2.k7", 192, 192, 192, 7, 9, 1280),
])
def test_small_calls_take_the_small_kernel_and_loaded_steps_do_not(layer):
    name, c_in, n_cols, c_out, taps, d, positions = layer
    kw = dict(c_in=c_in, n_cols=n_cols, c_out=c_out, taps=taps, dilation=d,
              left_pad=1 if taps == 2 else None)
    one = plan_shapes(batch=1, length=positions, **kw)
    assert one.kernel == N.CONV_KERNEL_SMALL and one.configs == 9
    assert plan_shapes(batch=64, length=positions * 3, **kw).kernel == N.CONV_KERNEL_DMA
    # E4M3 weights and operands activated while staged keep their kernels
    assert plan_shapes(batch=1, length=positions, fp8=True, **kw).kernel == N.CONV_KERNEL_DMA
    act = plan_shapes(batch=1, length=positions, in_activation=N.ACT_SNAKE, **kw)
    assert act.kernel == N.CONV_KERNEL_STAGED


def test_what_no_tile_serves_the_small_kernel_does_not_either():
    """The small kernel takes over calls that the large tiles serve, no others: many rows of two
    samples with a wide halo fit no k = 7 tile and stay refused."""
    kw = dict(batch=64, length=2, c_in=384, n_cols=384, c_out=384, taps=7, dilation=9)
    with pytest.raises(N.OmniCodecError, match="status 2"):
        plan_shapes(**kw)
    unit = plan_shapes(batch=1, length=1280, c_in=192, n_cols=192, c_out=192, taps=7, dilation=9,
                       fused_unit=True)
    assert unit.kernel == N.CONV_KERNEL_SMALL and unit.configs == 1
    loaded = plan_shapes(batch=64, length=3840, c_in=192, n_cols=192, c_out=192, taps=7,
                         dilation=9, fused_unit=True)
    assert loaded.kernel == N.CONV_KERNEL_FUSED_UNIT


@pytest.mark.parametrize("c_in,n_cols", [(96, 192), (192, 192), (192, 768), (384, 384)])
def test_one_tap_small_calls_start_every_workgroup_at_once(c_in, n_cols):
    """A CU holds eight waves of the one-tap small kernel; a call whose workgroups are more starts
    some of them after the others' end and is slower than the LDS-DMA tiles."""
    for positions in range(100, 12000, 100):
        plan = plan_shapes(batch=1, length=positions, c_in=c_in, n_cols=n_cols, c_out=n_cols, taps=1)
        if plan.kernel == N.CONV_KERNEL_SMALL:
            waves = (1, 2, 4)[(plan.config - 1) % 3]
            assert -(-plan.workgroups // 256) * waves <= 8, (positions, plan)


@pytest.mark.parametrize("positions", [2049, 2500, 2905, 3000])
def test_deep_one_tap_layers_take_the_tile_of_192_positions(positions):
    """1536 -> 1536 columns, us: 96 x 192 28.4, the smaller list's 96 x 256 30.0 (up to 2 048
    positions one round of its 96 x 128 tiles, 22.7)."""
    plan = plan_shapes(batch=1, length=positions, c_in=1536, n_cols=1536, c_out=1536, taps=1)
    assert plan.kernel == N.CONV_KERNEL_DMA and plan.config == 3


@pytest.mark.parametrize("batch,length,form", [
    # the form measured fastest of the four (us: sweep / 384 / 256 / 128 rows)
    (1, 310, N.STACK_FORM_ROWS128),       # 84 / 52 / 41 / 29
    (8, 1500, N.STACK_FORM_ROWS256),      # 131 / 55 / 43 / 56
    (16, 7680, N.STACK_FORM_ROWS384),     # 131 / 106 / 117 / 275
    (48, 2371, N.STACK_FORM_SWEEP),       # 100 / 106 / 118 / 274
    (100, 2371, N.STACK_FORM_SWEEP),      # 180 / 209 / 228 / 556
    (128, 1000, N.STACK_FORM_SWEEP),      # 102 / 106 / 122 / 299
    (223, 400, N.STACK_FORM_SWEEP),       # 86 / 102 / 116 / 230
    (174, 2000, N.STACK_FORM_ROWS384),    # 282 / 265 / 340 / 653
    (512, 1000, N.STACK_FORM_SWEEP),      # 310 / 405 / 471 / 1137
    (1, 480000, N.STACK_FORM_SWEEP),      # 292 / 365 / 405 / 909
    (64, 23040, N.STACK_FORM_SWEEP), (8, 60001, N.STACK_FORM_SWEEP),
    (64, 12, N.STACK_FORM_ROWS384), (1, 300, N.STACK_FORM_ROWS384),  # whole rows
])
def test_the_stack_takes_its_fastest_form(batch, length, form):
    final = 7 if batch % 2 == 0 else 0
    chosen, workgroups = plan_stack_shapes(batch=batch, length=length, dilations=(1, 3, 9),
                                           final_taps=final)
    assert chosen == form
    # the named form is the same plan
    assert plan_stack_shapes(batch=batch, length=length, dilations=(1, 3, 9), final_taps=final,
                             form=form) == (chosen, workgroups)


def test_a_stack_form_that_cannot_hold_the_call_is_refused():
    with pytest.raises(N.OmniCodecError):
        plan_stack_shapes(batch=1, length=1000, dilations=(1,), form=N.STACK_FORM_ROWS128 + 1)
    for kw in (dict(length=300, dilations=(1, 3, 9), form=N.STACK_FORM_SWEEP),      # one tile
               dict(length=2000, dilations=(1, 1, 3, 9), form=N.STACK_FORM_SWEEP),  # four units
               dict(length=2000, dilations=(10,), form=N.STACK_FORM_SWEEP),         # halo past the guard
               dict(length=2000, dilations=(10, 9), form=N.STACK_FORM_ROWS128)):    # 114 halo rows of 128
        with pytest.raises(N.OmniCodecError) as e:
            plan_stack_shapes(batch=1, **kw)
        assert e.value.status == N.UNSUPPORTED
