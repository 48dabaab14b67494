"""``_native.stream_handle`` is the current stream's handle for every way of naming the device: on
the default stream, inside a side stream, nested, on another thread (which starts on the default
stream) and under a graph capture, where a launch on any other stream would break the capture."""

from __future__ import annotations

import threading

import pytest
import torch

from sglang_omni_amd import _native as N

pytestmark = pytest.mark.gpu


def _devices():
    return [None, torch.device("cuda"), torch.device("cuda", torch.cuda.current_device()),
            torch.empty(0, device="cuda").device]


@pytest.mark.parametrize("which", range(4))
def test_current_stream(gpu, which):
    device = _devices()[which]
    default = torch.cuda.default_stream().cuda_stream
    assert N.stream_handle(device) == default
    outer, inner = torch.cuda.Stream(), torch.cuda.Stream()
    seen = []
    with torch.cuda.stream(outer):
        assert N.stream_handle(device) == outer.cuda_stream != default
        with torch.cuda.stream(inner):
            assert N.stream_handle(device) == inner.cuda_stream
        thread = threading.Thread(target=lambda: seen.append(N.stream_handle(device)))
        thread.start()
        thread.join()
        assert N.stream_handle(device) == outer.cuda_stream
    assert seen == [default] and N.stream_handle(device) == default

    x = torch.ones(8, device="cuda")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=outer):
        assert N.stream_handle(device) == outer.cuda_stream
        x.add_(1)
    torch.cuda.synchronize()


def test_cpu_device_is_refused(gpu):
    with pytest.raises(ValueError):
        N.stream_handle(torch.device("cpu", 0))
    with pytest.raises(N.OmniCodecError, match="GPU tensors"):
        N.require_device(torch.empty(1, device="cuda"), None, torch.empty(1))
