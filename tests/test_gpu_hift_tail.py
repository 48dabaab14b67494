"""The iSTFT tail's own exp, sine and cosine over their ranges, and its frame windows at their edges,
against float64.

Bound: an output is a sum of 4 x 18 products of magnitude * cos / sin with the basis over the
envelope, each factor within 4 float32 roundings (exp, sine of a sine, product) and the sums within
72 more, relative to the sum of the absolute terms."""

from __future__ import annotations

import pytest
import torch

from oracle import codec_oracle as O
from sglang_omni_amd.kernels.hift import HiftStft, overlap_add_inverse

pytestmark = pytest.mark.gpu


def parts(h):
    h = h.double()
    mag, phase = torch.exp(h[..., :9]).clamp(max=100.0), torch.sin(h[..., 9:18])
    return (mag * torch.cos(phase)).transpose(1, 2), (mag * torch.sin(phase)).transpose(1, 2)


# one frame more than a workgroup's window of quads, one less, ragged, one sample quad
@pytest.mark.parametrize("frames", [2, 255, 256, 257, 258, 511, 514, 1003])
@pytest.mark.parametrize("phase_scale", [1.0, 300.0, 3e4, 1e6])
@pytest.mark.parametrize("layout", ["packed", "wide", "unaligned"])
def test_tail_against_float64(gpu, frames, phase_scale, layout):
    gen = torch.Generator().manual_seed(frames)
    h = torch.randn(3, frames, 18, generator=gen)
    h[..., :9] = h[..., :9] * 0.8 - 4.0
    h[..., 9:] *= phase_scale
    h[0, :, 0] = torch.linspace(-140.0, 2.0, frames)  # magnitudes down to zero
    h[1, :, 9] = torch.pi * torch.arange(frames).float()  # sines near zero
    st = HiftStft(O.hann_window(16), 4, device=gpu)
    hd = h.to(gpu)
    if layout == "wide":  # rows of 20 channels, the last two not read
        hd = torch.cat([hd, torch.full((3, frames, 2), float("nan"), device=gpu)], dim=2)
    elif layout == "unaligned":  # a view whose first element is 4 bytes past an 8-byte boundary
        flat = torch.empty(3 * frames * 18 + 1, device=gpu)
        flat[1:] = hd.reshape(-1)
        hd = flat[1:].view(3, frames, 18)
    re, im = parts(h)
    want = O.istft_reference(re, im, O.hann_window(16), 16, 4).clamp(-0.99, 0.99)
    scale = float(torch.maximum(re.abs(), im.abs()).amax())
    got = st.tail(hd).cpu()
    assert got.shape == want.shape
    err = (got.double() - want).abs().max().item()
    # 18 components of at most `scale`, basis at most 2 / 16, over 4 frames and an envelope >= 1.49
    assert err <= (4 + 72) * 2.0 ** -24 * 4 * 18 * scale * (2 / 16) / 1.49
    # the inverse over the same parts, rounded to float32 first
    inv = overlap_add_inverse(re.float().contiguous().to(gpu), im.float().contiguous().to(gpu),
                              st.inverse_basis, st.squared_window, 4).cpu()
    full = O.istft_reference(re, im, O.hann_window(16), 16, 4)
    assert (inv.double() - full).abs().max().item() <= 74 * 2.0 ** -24 * 9 * scale / 1.49


def test_tail_at_the_ends_of_the_range(gpu):
    """Infinite magnitudes clip, vanishing ones are zero, and a NaN or infinite phase marks the
    samples of its frame's window and no other."""
    st = HiftStft(O.hann_window(16), 4, device=gpu)
    h = torch.full((1, 400, 18), -3.0)
    h[..., 9:] = 0.5
    h[0, 100, 3], h[0, 101, 4], h[0, 102, 5] = float("inf"), float("-inf"), 1e30
    re, im = parts(h)
    want = O.istft_reference(re, im, O.hann_window(16), 16, 4).clamp(-0.99, 0.99)
    torch.testing.assert_close(st.tail(h.to(gpu)).cpu().double(), want, rtol=1e-5, atol=1e-5)
    clean = st.tail(h.to(gpu)).cpu()[0]
    for bad in (float("nan"), float("inf")):
        h[0, 200, 12] = bad
        got = st.tail(h.to(gpu)).cpu()[0]
        # frame 200 covers samples 792 .. 807, and the clamp turns their NaN into its lower limit
        inside = torch.zeros(got.numel(), dtype=torch.bool)
        inside[792:808] = True
        assert torch.equal(got[~inside], clean[~inside])
        assert bool((got[inside] == -0.99).all()) and not bool((clean[inside] == -0.99).any())


def library_tail(st, h, clip, limit):
    """The tail with the library's exp, sin and cos, through the same inverse transform."""
    mag, phase = torch.exp(h[..., :9]).clamp(max=clip), torch.sin(h[..., 9:])
    re, im = ((mag * f(phase)).transpose(1, 2).contiguous() for f in (torch.cos, torch.sin))
    return overlap_add_inverse(re, im, st.inverse_basis, st.squared_window, 4).clamp(-limit, limit)


@pytest.mark.parametrize("low,high", [(-0.8, 0.8), (1.2, 2.0), (4.2, 5.2), (-9.0, 9.0),
                                      (-300.0, 300.0), (-3e4, 3e4)])
@pytest.mark.parametrize("bin_", [0, 3, 8])
@pytest.mark.parametrize("log_mag", [0.0, -6.0])
def test_tail_is_no_further_from_float64_than_the_library(gpu, low, high, bin_, log_mag):
    """One bin of every fourth frame alone, so a sample is that bin's exp, sin and cos, two products,
    a sum and a division: the mean square error against float64 is no larger than with the
    library's functions in their place (2 % for the draw: 2^18 samples whose errors are mostly the
    common products)."""
    frames = 2 ** 16 + 1
    gen = torch.Generator().manual_seed(bin_ + int(abs(low) * 10))
    h = torch.full((1, frames, 18), -200.0)
    h[..., 9:] = torch.rand(1, frames, 9, generator=gen) * (high - low) + low
    h[0, ::4, bin_] = log_mag - 2.0 * torch.rand((frames + 3) // 4, generator=gen) * abs(log_mag)
    st = HiftStft(O.hann_window(16), 4, device=gpu)
    re, im = parts(h)
    basis, squared = st.inverse_basis.double().cpu(), st.squared_window.double().cpu()
    frame = torch.einsum("bcf,ct->bft", torch.cat([re, im], 1), basis)[0]
    want = torch.zeros(frames + 3, 4, dtype=torch.float64)
    env = torch.zeros_like(want)
    for o in range(4):
        want[o:o + frames] += frame[:, 4 * o:4 * o + 4]
        env[o:o + frames] += squared[4 * o:4 * o + 4]
    want = (want / env).flatten()[8:8 + 4 * (frames - 1)]

    def error(y):
        return (y.double().cpu()[0] - want).square().mean().sqrt().item()

    got = error(st.tail(h.to(gpu)))
    assert got > 0 and got <= 1.02 * error(library_tail(st, h.to(gpu), 100.0, 0.99))


def test_tail_keeps_the_smallest_magnitudes(gpu):
    """Magnitudes below the smallest normal number (2^-126, exp(-87.4)) down to the smallest of all:
    each component within half a unit of 2^-149 and a rounding of 2^-24, 16 of them and the division."""
    st = HiftStft(O.hann_window(16), 4, device=gpu)
    h = torch.full((1, 601, 18), -200.0)
    h[..., 9:] = 0.25
    h[0, ::4, 0] = torch.linspace(-102.0, -80.0, 151)
    re, im = parts(h)
    want = O.istft_reference(re, im, O.hann_window(16), 16, 4)[0].double()
    got = st.tail(h.to(gpu)).cpu()[0].double()
    lib = library_tail(st, h.to(gpu), 100.0, 0.99).cpu()[0].double()
    assert (got - want).abs().max() <= (lib - want).abs().max() + 2.0 ** -149
    assert bool(((got - want).abs() <= 2.0 ** -22 * want.abs() + 3 * 2.0 ** -149).all())


def test_a_few_frames_cost_the_tail_no_full_window(gpu):
    """A workgroup ran exp, sine and cosine over its whole window of 259 frames however few the row
    has: five frames took the tail 1.27 times the inverse's time, now 0.92 (each the least of ten
    replays of 20 calls)."""
    st = HiftStft(O.hann_window(16), 4, device=gpu)
    h = torch.randn(3, 5, 18, device=gpu)
    re, im = (torch.randn(3, 9, 5, device=gpu) for _ in range(2))
    graphs = []
    side = torch.cuda.Stream()
    for run in (lambda: st.tail(h),
                lambda: overlap_add_inverse(re, im, st.inverse_basis, st.squared_window, 4)):
        with torch.cuda.stream(side):
            run()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            kept = [run() for _ in range(20)]
        graphs.append((graph, kept))
    start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    best = [float("inf")] * 2
    for _ in range(10):
        for i, (graph, _) in enumerate(graphs):
            start.record()
            graph.replay()
            end.record()
            torch.cuda.synchronize()
            best[i] = min(best[i], start.elapsed_time(end))
    assert best[0] <= 1.1 * best[1], best
