"""The stream that kernels are launched on is torch's current one, in every context that changes it."""
import threading

import pytest
import torch

from distributed_llms_amd.ops.stream import current_stream


@pytest.mark.gpu
def test_handle_follows_the_current_stream(cuda):
    want = lambda: torch.cuda.current_stream().cuda_stream
    assert current_stream() == want()
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        assert current_stream() == want() == s.cuda_stream
        seen = []
        t = threading.Thread(target=lambda: seen.append((current_stream(), want())))
        t.start()
        t.join()
        assert seen[0][0] == seen[0][1] != s.cuda_stream            # a stream is current for one thread
        x = torch.zeros(8, device="cuda")
        s.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            assert current_stream() == want() != s.cuda_stream      # the capture's own
            x.add_(1)
    assert current_stream() == want()
