"""Scratch of captured calls: a graph keeps writing to what it was captured with, so that must not be the shared buffer."""
import pytest
import torch

from fastgl import _lib as L
from fastgl import ops

pytestmark = pytest.mark.gpu


def test_captured_calls_keep_their_scratch(cuda):
    a, b = torch.randn(30000, 100, device=cuda), torch.randn(30000, 64, device=cuda)
    big = torch.randn(60000, 256, device=cuda)
    want = ops.weight_grad(a, b)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        shared = dict(L._workspaces)
        got = ops.weight_grad(a, b)
        assert dict(L._workspaces) == shared, "a captured call took (and may have replaced) the shared scratch"
    for _ in range(3):
        got.zero_()
        graph.replay()
        ops.weight_grad(big, big)  # eager work with larger scratch between the replays
        torch.cuda.synchronize()
        assert torch.equal(got, want)
