"""``omni_conv1d_general`` on the matrix cores, against the float64 conv of the same operands, over
the forms it accepts: dtypes, groups, strides, dilations, padding, channel counts on and off the
16-byte grid, strided views, lengths at the tiles' edges (32 and 128 positions; 32, 64 and 96
columns), and values at the ends of the range.

Bounds: an output is a float32 sum of exact (2-byte) or once-rounded (float32) products, so its
error is below (K + 2) 2^-24 sum |x w| (K products and the bias, any order), plus one rounding to
the dtype."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from sglang_omni_amd.utils.channels_last_conv import (
    _general,
    channels_last_conv1d,
    channels_last_conv_transpose1d,
    channels_last_weight,
)

pytestmark = pytest.mark.gpu

EPS = {torch.float32: 2.0 ** -24, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def conv64(x, w, b, *, groups, stride, dilation, pad, transposed, length):
    """The first ``length`` outputs of the float64 conv (left padding only) of x [B, L, C]."""
    x, w = x.double().cpu().transpose(1, 2), w.double().cpu()
    b = None if b is None else b.double().cpu()
    if transposed:
        y = F.conv_transpose1d(x, w, b, stride=stride, dilation=dilation, groups=groups)
        y = F.pad(y, (0, max(0, length + pad - y.shape[2])))
        if b is not None:  # positions past the last input's reach hold the bias
            full = (x.shape[2] - 1) * stride + dilation * (w.shape[2] - 1) + 1
            y[:, :, full:] = b[:, None]
        return y[:, :, pad:pad + length].transpose(1, 2)
    reach = (w.shape[2] - 1) * dilation
    right = max(0, (length - 1) * stride + reach + 1 - pad - x.shape[2])
    y = F.conv1d(F.pad(x, (pad, right)), w, b, stride=stride, dilation=dilation, groups=groups)
    return y[:, :, :length].transpose(1, 2)


def check(got, x, w, b, **kw):
    want = conv64(x, w, b, length=got.shape[1], **kw)
    size = conv64(x.abs(), w.abs(), None if b is None else b.abs(), length=got.shape[1], **kw)
    terms = w.shape[2] * (w.shape[0] // kw["groups"] if kw["transposed"] else w.shape[1])
    bound = (terms + 2) * 2.0 ** -24 * size + EPS[got.dtype] * want.abs() + 2.0 ** -25
    err = (got.double().cpu() - want).abs()
    assert bool((err <= bound).all()), f"worst {float((err / bound).max()):.2f} of the bound"


def draw(gpu, dtype, batch, length, c_in, c_out, taps, groups, transposed, seed=0):
    g = torch.Generator().manual_seed(seed)
    shape = (c_in, c_out // groups, taps) if transposed else (c_out, c_in // groups, taps)
    x = torch.randn(batch, length, c_in, generator=g).to(dtype).to(gpu)
    w = (torch.randn(shape, generator=g) * 0.1).to(dtype).to(gpu)
    b = torch.randn(c_out, generator=g).to(dtype).to(gpu)
    return x, w, b


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("batch,length,c_in,c_out,taps,groups,stride,dilation,pad,transposed", [
    (2, 4801, 192, 192, 7, 1, 1, 3, 0, False),   # 96-column, 128-position tiles, an odd tail
    (1, 700, 64, 64, 11, 1, 1, 5, 25, False),    # more taps than a stage, left padding
    (3, 129, 40, 48, 3, 1, 1, 1, 1, False),      # channels past whole chunks
    (2, 300, 17, 33, 5, 1, 2, 2, 3, False),      # odd channels: elements one by one; strided
    (1, 2000, 24, 16, 20, 1, 8, 1, 6, False),    # stride past the wide tile's rows
    (2, 31, 64, 96, 41, 2, 1, 1, 40, False),     # groups, many taps, fewer rows than a tile
    (4, 33, 96, 24, 1, 1, 1, 1, 0, False),
    (2, 2003, 256, 128, 11, 1, 5, 1, 3, True),   # the vocoder's upsampler, an odd length
    (1, 50, 64, 32, 8, 1, 4, 1, 2, True),
    (2, 37, 32, 48, 7, 1, 4, 2, 0, True),        # dilation sharing a factor with the stride
    (1, 19, 36, 20, 3, 1, 6, 3, 1, True),        # phases without taps: bias only
    (2, 65, 64, 64, 4, 4, 2, 1, 1, True),        # grouped
    (1, 400, 16, 128, 3, 1, 1, 1, 1, True),
])
def test_every_form_matches_the_float64_conv(gpu, dtype, batch, length, c_in, c_out, taps, groups,
                                             stride, dilation, pad, transposed):
    x, w, b = draw(gpu, dtype, batch, length, c_in, c_out, taps, groups, transposed)
    if transposed:
        out = (length - 1) * stride + dilation * (taps - 1) + 1 - pad
    else:
        out = (length + pad - (taps - 1) * dilation - 1) // stride + 1
    kw = dict(groups=groups, stride=stride, dilation=dilation, transposed=transposed)
    for bias in (b, None):
        got = _general(x, w, bias, c_out=c_out, pad_left=pad, length_out=out, **kw)
        check(got, x, w, bias, pad=pad, **kw)
    # the module's strides, a channels-last copy and a view into longer rows give the same bits
    cl = w.transpose(1, 2).contiguous().transpose(1, 2)
    assert torch.equal(_general(x, cl, b, c_out=c_out, pad_left=pad, length_out=out, **kw),
                       _general(x, w, b, c_out=c_out, pad_left=pad, length_out=out, **kw))
    wide = torch.full((batch, length + 3, c_in + 5), float("nan"), dtype=dtype, device=gpu)
    wide[:, 2:2 + length, 1:1 + c_in] = x
    assert torch.equal(
        _general(wide[:, 2:2 + length, 1:1 + c_in], w, b, c_out=c_out, pad_left=pad, length_out=out,
                 **kw),
        _general(x, w, b, c_out=c_out, pad_left=pad, length_out=out, **kw))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_small_values_are_kept_and_infinities_stay_where_they_reach(gpu, dtype):
    """Subnormal operands enter the products as they are, and an infinite or NaN input marks the
    outputs its taps reach and no other."""
    x, w, b = draw(gpu, dtype, 1, 200, 32, 32, 3, 1, False)
    tiny = x * (2.0 ** -16 if dtype == torch.float16 else 2.0 ** -120)
    big = w * (2.0 ** 13 if dtype == torch.float16 else 2.0 ** 100)
    conv = torch.nn.Conv1d(32, 32, 3).to(gpu).to(dtype)
    got = channels_last_conv1d(tiny, conv, big, None, 198)
    want = conv64(tiny, big, None, groups=1, stride=1, dilation=1, pad=0, transposed=False,
                  length=198)
    torch.testing.assert_close(got.double().cpu(), want, rtol=2e-3 if dtype == torch.float16 else 1e-5,
                               atol=float(want.abs().mean()) * 1e-3)
    x[0, 100, 5], x[0, 160, 7] = float("inf"), float("nan")
    bad = ~torch.isfinite(channels_last_conv1d(x, conv, w, b, 198)).all(dim=2)[0].cpu()
    assert bad.nonzero().flatten().tolist() == [98, 99, 100, 158, 159, 160]
    up = torch.nn.ConvTranspose1d(32, 32, 4, stride=3).to(gpu).to(dtype)
    bad = ~torch.isfinite(channels_last_conv_transpose1d(x, up, channels_last_weight(up),
                                                         up.bias)).all(dim=2)[0].cpu()
    assert bad.nonzero().flatten().tolist() == [300, 301, 302, 303, 480, 481, 482, 483]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("length,taps,groups,stride,dilation,pad,transposed", [
    (300, 7, 1, 1, 3, 11, False),   # both ends of a row, inside a stage of taps
    (129, 20, 2, 1, 1, 10, False),  # several stages of taps
    (5, 7, 1, 1, 1, 3, False),      # every output is near an end
    (200, 5, 1, 2, 2, 5, False),
    (100, 11, 1, 5, 1, 3, True),
    (40, 8, 2, 4, 3, 2, True),
])
def test_a_tap_outside_the_row_adds_nothing_whatever_its_weight(gpu, dtype, bad, length, taps, groups,
                                                                 stride, dilation, pad, transposed):
    """An infinite or NaN weight marks the outputs that its tap reaches inside the row; the others
    are those of a zero weight in its place."""
    x, w, b = draw(gpu, dtype, 2, length, 32, 48, taps, groups, transposed)
    reach = (taps - 1) * dilation
    out = ((length - 1) * stride + reach + 1 if transposed else (length + 2 * pad - reach - 1) // stride + 1)
    kw = dict(groups=groups, stride=stride, dilation=dilation, transposed=transposed)
    place = dict(c_out=48, pad_left=pad, length_out=out)
    i, missed = torch.arange(out), 0
    for tap in (0, taps // 2, taps - 1):
        if transposed:
            at = i + pad - tap * dilation
            reached = (at % stride == 0) & (at >= 0) & (at < length * stride)
        else:
            at = i * stride + tap * dilation - pad
            reached = (at >= 0) & (at < length)
        zero, one = w.clone(), w.clone()
        column = (3, 5, tap)  # output channel 5 of group 0 (transposed), output channel 3
        zero[column], one[column] = 0.0, bad
        channel = 5 if transposed else 3
        want, got = _general(x, zero, b, **place, **kw), _general(x, one, b, **place, **kw)
        reached = reached.to(gpu)
        missed += int((~reached).sum())
        assert not bool(torch.isfinite(got[:, reached, channel]).any())
        got[:, reached, channel] = want[:, reached, channel]
        check(got, x, zero, b, pad=pad, **kw)
        got[:, :, channel] = want[:, :, channel]
        assert torch.equal(got, want)
    assert missed > 0  # outputs that a tap does not reach


# forms on both sides of the line between the matrix cores and one thread per output
LINE = [
    (58, 2, 1536, 320, 2, 64, 8, 1, 0, True),   # 64 groups, 8 phases, 2 taps: tiny workgroups
    (62, 3, 128, 1536, 1, 32, 8, 3, 0, True),
    (46, 9, 512, 128, 2, 32, 8, 1, 3, True),
    (21, 51, 192, 128, 1, 32, 4, 1, 0, False),
    (3, 171, 768, 256, 1, 64, 1, 1, 0, False),
    (40, 8, 64, 64, 3, 16, 1, 1, 2, False),
    (9, 300, 48, 48, 4, 2, 2, 1, 1, True),
    (12, 40, 96, 96, 7, 1, 1, 3, 6, False),
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("batch,length,c_in,c_out,taps,groups,stride,dilation,pad,transposed", LINE)
def test_a_row_does_not_depend_on_the_rows_beside_it(gpu, dtype, batch, length, c_in, c_out, taps,
                                                     groups, stride, dilation, pad, transposed):
    """The kernel is chosen without regard to the batch, so a row has the same bits alone."""
    x, w, b = draw(gpu, dtype, batch, length, c_in, c_out, taps, groups, transposed)
    reach = dilation * (taps - 1)
    out = (length - 1) * stride + reach + 1 - pad if transposed else (length + pad - reach - 1) // stride + 1
    kw = dict(groups=groups, stride=stride, dilation=dilation, transposed=transposed)
    got = _general(x, w, b, c_out=c_out, pad_left=pad, length_out=out, **kw)
    check(got, x, w, b, pad=pad, **kw)
    for rows in (slice(0, 1), slice(batch - 1, batch), slice(1, 3)):
        assert torch.equal(_general(x[rows], w, b, c_out=c_out, pad_left=pad, length_out=out, **kw),
                           got[rows])


@pytest.mark.parametrize("batch,length,c_in,c_out,taps,groups,stride,dilation,pad,transposed", LINE[:3])
def test_many_small_groups_are_not_a_workgroup_each(gpu, batch, length, c_in, c_out, taps, groups,
                                                    stride, dilation, pad, transposed):
    """As matrix-core tiles of a few outputs each these took 7 to 20 times a single row's time (23 and
    more us); one thread per output takes 1.5 to 3 times (7 to 12 us)."""
    def microseconds(rows):
        x, w, b = draw(gpu, torch.float32, rows, length, c_in, c_out, taps, groups, transposed)
        out = (length - 1) * stride + dilation * (taps - 1) + 1 - pad
        run = lambda: _general(x, w, b, c_out=c_out, pad_left=pad, length_out=out, groups=groups,
                               stride=stride, dilation=dilation, transposed=transposed)
        side = torch.cuda.Stream()
        with torch.cuda.stream(side):
            run()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            kept = [run() for _ in range(20)]
        start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        best = float("inf")
        for _ in range(10):
            start.record()
            graph.replay()
            end.record()
            torch.cuda.synchronize()
            best = min(best, start.elapsed_time(end) * 1e3 / len(kept))
        return best

    assert microseconds(batch) <= 4.5 * microseconds(1)
