"""Blocks whose tiles (of 8192 rows from 524288 rows on, 2048 below) are partly alike (taken as they come) and partly not (taken in order of
length), with two, four and eight rows to a wave: rows of up to 128 entries against the same rows in one launch, bit for bit, the longer ones against float64 sums."""
import pytest
import torch

from fastgl import ops

pytestmark = pytest.mark.gpu

TILE = 8192


def _lens(kinds, tail, gen):
    parts = []
    for kind in kinds:
        if kind == "alike":
            parts.append(torch.full((TILE,), 8))
        elif kind == "empty":
            parts.append(torch.zeros(TILE, dtype=torch.int64))
        else:
            lens = torch.where(torch.rand(TILE, generator=gen) < 0.8, 0, torch.randint(1, 100, (TILE,), generator=gen))
            lens[:: 500] = torch.randint(120, 700, (lens[::500].numel(),), generator=gen)
            parts.append(lens)
    return torch.cat(parts)[:len(kinds) * TILE - tail].long()


@pytest.mark.parametrize("dim,dtype", [(128, torch.float32), (64, torch.float32), (40, torch.bfloat16), (200, torch.bfloat16), (33, torch.float32)])
@pytest.mark.parametrize("tail,times", [(0, 3), (1, 3), (2047, 3), (TILE - 1, 3), (1, 11)])
def test_tiles_in_order_and_as_they_come(cuda, dim, dtype, tail, times):
    print("row tiles", dim, dtype, tail, times, flush=True)
    gen = torch.Generator().manual_seed(dim + tail)
    lens = _lens(["alike", "skewed", "empty", "skewed", "alike", "alike"] * times + ["skewed"], tail, gen)
    n, n_cols = lens.numel(), 60_000
    ptr = torch.zeros(n + 1, dtype=torch.int64)
    ptr[1:] = torch.cumsum(lens, 0)
    assert int(ptr[-1]) >= 1 << 19 and n >= 1 << 17
    idx = torch.randint(0, n_cols, (int(ptr[-1]),), generator=gen, dtype=torch.int32)
    x = torch.randn((n_cols, dim), generator=gen).to(dtype)
    d_ptr, d_idx, d_x = ptr.int().to(cuda), idx.to(cuda), x.to(cuda)
    plain = ops.aggregate(d_ptr, d_idx, d_x, mode="sum", zero_policy="zeros", n_rows=n, mapping="row")
    short = (lens <= 128).to(cuda)
    longest = torch.tensor([int(lens.max())], dtype=torch.int32, device=cuda)
    for kw in ({}, dict(longest_row=longest)):
        out = torch.full((n, dim), 7.0, dtype=dtype, device=cuda)
        ops.aggregate(d_ptr, d_idx, d_x, mode="sum", zero_policy="zeros", n_rows=n, out=out, **kw)
        assert torch.equal(out[short], plain[short])
        for r in torch.nonzero(lens > 128).flatten()[::7 * times].tolist():
            rows = x[idx[ptr[r]:ptr[r + 1]].long()].double()
            # (sums of up to 700 entries in two levels: far below n 2^-24 of the sum of magnitudes; bf16 results are rounded once more)
            bound = int(lens[r]) * 2.0 ** -24 * rows.abs().sum(0) + (rows.sum(0).abs() * 2.0 ** -8 if dtype == torch.bfloat16 else 0)
            assert bool(((out[r].cpu().double() - rows.sum(0)).abs() <= bound).all())
    # no row is long, which the device knows and the host does not: every row is this launch's, in order or not
    few = lens.clamp(max=128)
    ptr[1:] = torch.cumsum(few, 0)
    d_ptr, none = ptr.int().to(cuda), torch.zeros(1, dtype=torch.int32, device=cuda)
    d_idx = d_idx[:int(ptr[-1])]
    assert d_idx.numel() >= 1 << 19
    got = ops.aggregate(d_ptr, d_idx, d_x, mode="mean", zero_policy="zeros", n_rows=n, longest_row=none)
    assert torch.equal(got, ops.aggregate(d_ptr, d_idx, d_x, mode="mean", zero_policy="zeros", n_rows=n, mapping="row"))
