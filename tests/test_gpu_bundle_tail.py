"""Bundled rows (a transposed block's short lists) around the length that leaves a list to the second launch, against float64: lists of 47,
48, 49 and 128, 129 entries alone in their bundle and next to each other, at its ends, with the longest length known to the host or not."""
import pytest
import torch

from fastgl import _lib as L
from fastgl import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["sum", "colmean", "edge"])
@pytest.mark.parametrize("dim,dtype", [(64, torch.float32), (100, torch.float32), (256, torch.float32), (300, torch.float32), (128, torch.bfloat16),
                                       (600, torch.bfloat16)])
def test_lists_at_the_limit(cuda, mode, dim, dtype):
    print("bundle tail", mode, dim, dtype, flush=True)
    if mode == "edge" and dim not in (64, 128, 256):
        pytest.skip("rows whose vectors straddle heads are not bundled")
    gen = torch.Generator().manual_seed(dim)
    n_rows, n_cols = 16_385, 3000
    lens = torch.randint(0, 3, (n_rows,), generator=gen)
    for at, ls in ((0, (47, 48, 49, 50)), (8, (0, 49, 0, 0)), (16, (48, 48, 48, 48)), (24, (128, 0, 129, 1)), (33, (47,)), (35, (200, 200)), (n_rows - 1, (49,))):
        lens[at:at + len(ls)] = torch.tensor(ls)
    ptr = torch.zeros(n_rows + 1, dtype=torch.int64)
    ptr[1:] = torch.cumsum(lens, 0)
    nnz = int(ptr[-1])
    assert nnz <= 2 * n_rows
    idx = torch.randint(0, n_cols, (nnz,), generator=gen, dtype=torch.int32)
    x = torch.randn((n_cols, dim), generator=gen).to(dtype)
    kw, w = {}, torch.ones(nnz, 1, dtype=torch.float64)
    if mode == "colmean":
        norm = torch.randint(1, 20, (n_cols,), generator=gen, dtype=torch.int32)
        kw["col_norm"], w = norm.to(cuda), (1.0 / norm[idx.long()].double())[:, None]
    if mode == "edge":
        ew = torch.rand((nnz, 4), generator=gen)
        kw.update(edge_weight=ew.to(cuda), n_heads=4)
        w = ew.double().repeat_interleave(dim // 4, dim=1)
    rows = torch.repeat_interleave(torch.arange(n_rows), lens)
    want = torch.zeros((n_rows, dim), dtype=torch.float64).index_add_(0, rows, w * x[idx.long()].double())
    size = torch.zeros((n_rows, dim), dtype=torch.float64).index_add_(0, rows, (w * x[idx.long()].double()).abs())
    eps = 2.0 ** -23 * 24 * size + (want.abs() * 2.0 ** -8 if dtype == torch.bfloat16 else 0)  # (24 additions in a chain at most, and the weights)
    for longest in (None, 200, torch.tensor([200], dtype=torch.int32, device=cuda)):
        got = ops.aggregate(ptr.int().to(cuda), idx.to(cuda), x.to(cuda), mode=mode, zero_policy="zeros", n_rows=n_rows, longest_row=longest, **kw)
        assert b"bundled" in L.lib().fgl_aggregate_last_mapping() and b"long_rows" in L.lib().fgl_aggregate_last_mapping()
        assert bool(((got.cpu().double() - want).abs() <= eps).all())


@pytest.mark.parametrize("dim,dtype", [(300, torch.float32), (600, torch.bfloat16)])
@pytest.mark.parametrize("longest,second", [(49, False), (72, False), (73, True), (129, True)])
def test_wide_rows_with_a_longest_row_known_to_the_host(cuda, dim, dtype, longest, second):
    print("known longest", dim, dtype, longest, flush=True)
    gen = torch.Generator().manual_seed(longest)
    n_rows, n_cols = 16_385, 3000
    lens = torch.randint(0, 3, (n_rows,), generator=gen)
    lens[5::3001] = longest
    lens[-1] = longest
    ptr = torch.zeros(n_rows + 1, dtype=torch.int64)
    ptr[1:] = torch.cumsum(lens, 0)
    idx = torch.randint(0, n_cols, (int(ptr[-1]),), generator=gen, dtype=torch.int32)
    x = torch.randn((n_cols, dim), generator=gen).to(dtype)
    rows = torch.repeat_interleave(torch.arange(n_rows), lens)
    want, size = (torch.zeros((n_rows, dim), dtype=torch.float64).index_add_(0, rows, v) for v in (x[idx.long()].double(), x[idx.long()].double().abs()))
    got = ops.aggregate(ptr.int().to(cuda), idx.to(cuda), x.to(cuda), mode="sum", zero_policy="zeros", n_rows=n_rows, longest_row=longest)
    assert (b"long_rows" in L.lib().fgl_aggregate_last_mapping()) == second
    eps = 2.0 ** -24 * 73 * size + (want.abs() * 2.0 ** -8 if dtype == torch.bfloat16 else 0)  # (72 additions in a chain at most)
    assert bool(((got.cpu().double() - want).abs() <= eps).all())
