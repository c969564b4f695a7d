"""Long rows summed by one workgroup each: lists whose lengths lie at the edges of the lane groups' even shares, against float64."""
import pytest
import torch

from fastgl import _lib as L
from fastgl import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["sum", "edge"])
@pytest.mark.parametrize("dim,dtype", [(32, torch.float32), (64, torch.float32), (128, torch.float32), (256, torch.float32), (520, torch.float32),
                                       (256, torch.bfloat16)])
def test_lists_at_the_edges_of_the_shares(cuda, mode, dim, dtype):
    print("long row shares", mode, dim, dtype, flush=True)
    gen = torch.Generator().manual_seed(dim)
    n_cols = 2000
    lens = torch.tensor([129, 0, 143, 144, 145, 3, 255, 256, 257, 383, 385, 511, 512, 513, 1, 767, 769, 1023, 1024, 1025, 1536, 1537, 5000])
    n_rows = len(lens)
    ptr = torch.zeros(n_rows + 1, dtype=torch.int64)
    ptr[1:] = torch.cumsum(lens, 0)
    nnz = int(ptr[-1])
    idx = torch.randint(0, n_cols, (nnz,), generator=gen, dtype=torch.int32)
    x = torch.randn((n_cols, dim), generator=gen).to(dtype)
    kw, w = {}, torch.ones(nnz, 1, dtype=torch.float64)
    if mode == "edge":
        ew = torch.rand((nnz, 4), generator=gen)
        kw.update(edge_weight=ew.to(cuda), n_heads=4)
        w = ew.double().repeat_interleave(dim // 4, dim=1)
    terms = w * x[idx.long()].double()
    rows = [terms[ptr[r]:ptr[r + 1]] for r in range(n_rows)]
    want = torch.stack([t.sum(0) for t in rows])
    # a chunk's entries, a group's chunks and the groups: at most 64 + 10 + 64 additions after one another, two roundings of a product
    eps = torch.stack([t.abs().sum(0) for t in rows]) * 140 * 2.0 ** -24
    if dtype == torch.bfloat16:
        eps = eps + want.abs() * 2.0 ** -8
    got = ops.aggregate(ptr.int().to(cuda), idx.to(cuda), x.to(cuda), mode=mode, zero_policy="zeros", n_rows=n_rows, **kw)
    assert b"long_rows" in L.lib().fgl_aggregate_last_mapping()
    assert bool(((got.cpu().double() - want).abs() <= eps).all())
