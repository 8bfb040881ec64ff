"""The stream the Python binding launches on is torch's current one: default,
inside a stream context, in another thread, and under graph capture."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_current_stream(lib):
    import torch

    from longhornai_amd import ops

    def want():
        return torch.cuda.current_stream().cuda_stream

    assert ops.stream() == want()
    side = torch.cuda.Stream()
    seen = []
    with torch.cuda.stream(side):
        assert ops.stream() == want() == side.cuda_stream
        t = threading.Thread(target=lambda: seen.append((ops.stream(), want())))
        t.start()
        t.join()
    assert seen[0][0] == seen[0][1] != side.cuda_stream
    x = torch.linspace(-2, 3, 4096, device="cuda")
    q, s = ops.empty((4096,), np.int8), ops.empty((1,), np.float32)
    ops.run("lhq_q8_quantize_per_tensor", x, q, s, 4096)
    eager = ops.host(q).copy()
    q.zero_()
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g):
        assert ops.stream() == want()
        ops.run("lhq_q8_quantize_per_tensor", x, q, s, 4096)
    for _ in range(3):
        q.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(ops.host(q), eager)
