"""Scratch is each call's own: captured calls keep theirs, threads on one stream do not share, nothing is held between calls."""
import threading

import pytest
import torch

from fastgl import ops

pytestmark = pytest.mark.gpu


def test_captured_calls_keep_their_scratch(cuda):
    a, b = torch.randn(30000, 100, device=cuda), torch.randn(30000, 64, device=cuda)
    big = torch.randn(60000, 256, device=cuda)
    want = ops.weight_grad(a, b)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = ops.weight_grad(a, b)
    for _ in range(3):
        got.zero_()
        graph.replay()
        ops.weight_grad(big, big)  # eager work with larger scratch between the replays
        torch.cuda.synchronize()
        assert torch.equal(got, want)


def test_scratch_is_given_back(cuda):
    ptr = torch.arange(0, 3_000_001, 3, dtype=torch.int32, device=cuda)
    idx = torch.arange(3_000_000, dtype=torch.int32, device=cuda)
    torch.cuda.synchronize()
    held = torch.cuda.memory_allocated(cuda)
    ops.block_transpose(ptr, idx, 1_000_000, 3_000_000)
    ops.cal_deg(idx, 3_000_000)
    assert torch.cuda.memory_allocated(cuda) == held


def test_threads_on_one_stream(cuda):
    """A thread that counts and scans while another forms weight gradients, as a sampler beside a backward pass."""
    a, b = torch.randn(20000, 100, device=cuda), torch.randn(20000, 64, device=cuda)
    ids = torch.randint(0, 5000, (300_000,), dtype=torch.int32, device=cuda)
    want_w, want_d = ops.weight_grad(a, b), torch.bincount(ids.long(), minlength=5000).int()
    want_s = torch.cumsum(want_d, 0, dtype=torch.int32)
    wrong = []

    def run(what, call, want):
        for _ in range(200):
            if not torch.equal(call(), want):
                wrong.append(what)

    threads = [threading.Thread(target=run, args=t) for t in (("weight_grad", lambda: ops.weight_grad(a, b), want_w),
                                                              ("cal_deg", lambda: ops.cal_deg(ids, 5000), want_d),
                                                              ("exclusive_sum", lambda: ops.exclusive_sum(want_d)[1:], want_s))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
