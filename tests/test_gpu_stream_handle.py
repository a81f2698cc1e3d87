"""runtime.stream_handle() names the stream that is current at the call, not at
an earlier one, whichever way it became current."""
import ctypes

import pytest
import torch

from kvforge_amd import runtime as R

pytestmark = pytest.mark.gpu


def test_follows_the_current_stream():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    side = torch.cuda.Stream()

    def same(stream):
        want = ctypes.c_void_p(stream.cuda_stream).value
        return R.stream_handle().value == want == R.stream_handle(stream).value

    for _ in range(2):  # the first call looks the runtime up, later ones do not
        assert same(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            assert same(side)
        assert same(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        assert same(torch.cuda.current_stream())
        torch.zeros(1, device="cuda:0")
