"""The binding's default stream is torch's current stream: the default one, another, and one under
capture, each changed between calls."""
import pytest
import torch

from gpu_util import say

pytestmark = pytest.mark.gpu


def test_calls_follow_the_current_stream(pkg, dev):
    assert pkg._stream(None) == torch.cuda.current_stream().cuda_stream
    assert pkg._stream(7) == 7
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert pkg._stream(None) == side.cuda_stream != 0
        with torch.cuda.stream(torch.cuda.default_stream()):
            assert pkg._stream(None) == torch.cuda.default_stream().cuda_stream
        assert pkg._stream(None) == side.cuda_stream
    assert pkg._stream(None) == torch.cuda.current_stream().cuda_stream
    x = torch.randn(4096, device="cuda").to(torch.bfloat16)
    want = torch.empty_like(x)
    pkg.gelu_tanh(x, want)
    y = torch.zeros_like(x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    say("gelu on the capturing stream")
    with torch.cuda.graph(graph):
        pkg.gelu_tanh(x, y)
    torch.cuda.synchronize()
    assert not y.any(), "the call ran outside the capture"
    for _ in range(2):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y.view(torch.int16), want.view(torch.int16))
