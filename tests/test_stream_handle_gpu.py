"""The stream a call without `stream` is given (gpu): torch's current one, also
on a thread of its own and under graph capture."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


def test_stream_handle_is_the_current_stream(gpu):
    def both():
        return gpu.stream_handle(), torch.cuda.current_stream().cuda_stream

    torch.zeros(1, device="cuda")
    s = torch.cuda.Stream()
    got, want = both()
    assert got == want and got != s.cuda_stream
    assert gpu.stream_handle(s) == s.cuda_stream
    with torch.cuda.stream(s):
        assert both() == (s.cuda_stream, s.cuda_stream)
        other = []
        t = threading.Thread(target=lambda: other.append(both()))  # streams are per thread
        t.start()
        t.join()
        assert other[0][0] == other[0][1] != s.cuda_stream
    g = torch.cuda.CUDAGraph()
    x = torch.zeros(4, device="cuda")
    with torch.cuda.graph(g):
        x.add_(1)
        got, want = both()
    assert got == want != 0
