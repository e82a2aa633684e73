"""A sequence captured by the caller as the first one over a plan: the box is
declared outside the capture, and every replay gives the eager sweeps' bits."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["7pt", "25pt"])
def test_first_sequence_in_a_capture(gpu, name):
    bk = gpu
    st = bk.Stencil.make(name, seed=3)
    g = bk.PeriodicGrid((5, 6, 4))
    a, b, c, d = (bk.Brick(g.info, g.field_storage(0), 0) for _ in range(4))
    bk.sweep(st, b, a, g)  # builds the plan
    bk.device_sync()
    stream = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        bk.sweeps(st, a, b, g, 9, stream=stream.cuda_stream)
    for seed in (1, 2, 3):
        g.fill_uniform(a, seed)
        g.fill_uniform(c, seed)
        bk.device_sync()
        graph.replay()
        torch.cuda.synchronize()
        bk.sweeps(st, c, d, g, 9)
        bk.device_sync()
        x, y = b.storage.to_host()[g.interior], d.storage.to_host()[g.interior]
        assert np.array_equal(x.view(np.uint8), y.view(np.uint8))
