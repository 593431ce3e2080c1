"""Calls without a stream argument run on the caller's current stream: the
default one, a side stream, a stream under capture, another thread's."""
import threading

import pytest
import torch

import ikv

pytestmark = pytest.mark.gpu


def test_the_handle_is_the_current_streams(dev):
    def check():
        assert ikv._stream() == torch.cuda.current_stream().cuda_stream
        assert ikv._stream(None) == torch.cuda.current_stream().cuda_stream

    check()
    side, other = torch.cuda.Stream(), torch.cuda.Stream()
    assert ikv._stream(side) == side.cuda_stream
    x = torch.randn(3, 1024, device=dev)
    w = torch.ones(1024, device=dev)
    want = ikv.rms_norm(x, w, 1e-6)
    torch.cuda.synchronize()
    seen = []

    def elsewhere():
        check()  # a thread starts on the default stream
        with torch.cuda.stream(other):
            check()
            seen.append(ikv._stream())

    with torch.cuda.stream(side):
        check()
        t = threading.Thread(target=elsewhere)
        t.start()
        t.join()
        assert seen == [other.cuda_stream] and ikv._stream() == side.cuda_stream
        out = torch.zeros_like(x)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            check()
            ikv.rms_norm(x, w, 1e-6, out=out)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
    check()
