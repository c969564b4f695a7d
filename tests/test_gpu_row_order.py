"""Rows gathered in order of length (large blocks with long rows among them) against the same rows as they come: a row of up to 128
entries is the same sum, bit for bit, a longer one the same up to the order of its sum; at the sizes where the order starts and a tile ends."""
import pytest
import torch

import fastgl
from fastgl import ops

pytestmark = pytest.mark.gpu

K = 1 << 17


def _block(n_rows, n_cols, cuda, gen):
    lens = torch.randint(0, 9, (n_rows,), generator=gen)
    lens[torch.rand(n_rows, generator=gen) < 0.4] = 0
    lens[:: 1000] = torch.randint(60, 300, (lens[::1000].numel(),), generator=gen)  # on both sides of 128 and of the bins' end
    lens[1] = 700
    lens[-3:] = 0
    ptr = torch.zeros(n_rows + 1, dtype=torch.int64)
    ptr[1:] = torch.cumsum(lens, 0)
    return lens.to(cuda), ptr.int().to(cuda), torch.randint(0, n_cols, (int(ptr[-1]),), generator=gen, dtype=torch.int32).to(cuda)


@pytest.mark.parametrize("mode", ["sum", "mean", "gcn", "colmean"])
@pytest.mark.parametrize("n_rows,dim,dtype", [(K - 1, 64, torch.float32), (K, 64, torch.float32), (K + 1, 33, torch.float32), (18 * 8192, 100, torch.float32),
                                              (18 * 8192 + 1, 64, torch.bfloat16), (19 * 8192 - 1, 256, torch.bfloat16), (200_000, 128, torch.float32)])
def test_in_order_of_length(cuda, mode, n_rows, dim, dtype):
    print("row order", mode, n_rows, dim, dtype, flush=True)
    gen = torch.Generator().manual_seed(n_rows)
    n_cols = max(n_rows, 50_000)
    lens, ptr, idx = _block(n_rows, n_cols, cuda, gen)
    assert idx.numel() >= 1 << 18
    reps = -(-(1 << 19) // idx.numel())
    if reps > 1:  # (half a million entries and more: where long rows go in segments, and rows in order)
        lens = lens * reps
        ptr, idx = ptr * reps, torch.repeat_interleave(idx, reps)
    x = torch.randn((n_cols, dim), generator=gen).to(dtype).to(cuda)
    kw = {}
    if mode == "gcn":
        kw["row_norm"] = lens.clamp(min=1).int()
    if mode in ("gcn", "colmean"):
        kw["col_norm"] = torch.randint(1, 30, (n_cols,), generator=gen, dtype=torch.int32).to(cuda)
    for policy in ("self", "zeros"):
        got = ops.aggregate(ptr, idx, x, mode=mode, zero_policy=policy, n_rows=n_rows, **kw)
        plain = ops.aggregate(ptr, idx, x, mode=mode, zero_policy=policy, n_rows=n_rows, mapping="row", **kw)
        short = lens <= 128
        assert torch.equal(got[short], plain[short])
        assert float((got[~short].double() - plain[~short].double()).norm() / plain[~short].double().norm()) < (2e-6 if dtype == torch.float32 else 4e-3)
    fewer = torch.tensor([n_rows - 777], dtype=torch.int32, device=cuda)
    out = torch.full((n_rows, dim), 7.0, dtype=dtype, device=cuda)
    ops.aggregate(ptr, idx, x, mode=mode, zero_policy="zeros", n_rows=n_rows, n_rows_dev=fewer, out=out, **kw)
    keep = short[:n_rows - 777]
    assert torch.equal(out[:n_rows - 777][keep], plain[:n_rows - 777][keep]) and bool((out[n_rows - 777:] == 7).all())
