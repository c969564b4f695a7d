"""Long rows of large inputs: the segmented sums against a float64 product, at row lengths around the segment's edges."""
import pytest
import torch

from fastgl import _lib as L
from fastgl import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LENGTHS = [0, 1, 5, 127, 128, 129, 191, 192, 511, 512, 513, 1023, 1024, 1025, 4097, 70001]


def _block(n_cols):
    """Rows of the lengths above, the longest ones next to each other, padded with random ones to just over the least entry count."""
    gen = torch.Generator().manual_seed(7)
    lens = torch.cat([torch.tensor(LENGTHS * 3 + sorted(LENGTHS)), torch.randint(0, 700, (1500,), generator=gen)])
    ptr = torch.cat([torch.zeros(1, dtype=torch.int64), lens.cumsum(0)])
    assert int(ptr[-1]) >= L.AGG_SEG_MIN_ENTRIES
    idx = torch.randint(0, n_cols, (int(ptr[-1]),), generator=gen, dtype=torch.int32)
    return ptr.int().to(DEV), idx.to(DEV), lens.to(DEV)


@pytest.mark.parametrize("dim,dtype", [(3, torch.float32), (32, torch.float32), (37, torch.bfloat16), (64, torch.float32), (100, torch.float32),
                                       (256, torch.bfloat16), (300, torch.float32)])
@pytest.mark.parametrize("mode", ["sum", "mean", "gcn", "gcn_own", "colmean"])
def test_segments(dim, dtype, mode):
    n_cols = 20000
    ptr, idx, lens = _block(n_cols)
    n = int(lens.numel())
    gen = torch.Generator(device=DEV).manual_seed(dim)
    x = torch.randn((n_cols, dim), generator=gen, device=DEV).to(dtype)
    col = torch.randint(1, 50, (n_cols,), generator=gen, dtype=torch.int32, device=DEV)
    row = torch.randint(1, 50, (n,), generator=gen, dtype=torch.int32, device=DEV)
    kw = dict(mode=mode, zero_policy="zeros", col_norm=col if mode in ("gcn", "gcn_own", "colmean") else None, row_norm=row if mode == "gcn" else None)
    got = ops.aggregate(ptr, idx, x, **kw)
    assert torch.equal(got, ops.aggregate(ptr, idx, x, **kw)), "the sums depend on scheduling"
    deg = lens.clamp(min=1).double()
    rf = {"sum": torch.ones_like(deg), "colmean": torch.ones_like(deg), "mean": 1 / deg, "gcn_own": deg.rsqrt(), "gcn": row.double().rsqrt()}[mode]
    cf = {"gcn": col.double().rsqrt(), "gcn_own": col.double().rsqrt(), "colmean": 1 / col.double()}.get(mode, torch.ones(n_cols, dtype=torch.float64, device=DEV))
    dst = torch.repeat_interleave(torch.arange(n, device=DEV), lens)
    want, mag = torch.zeros((n, dim), dtype=torch.float64, device=DEV), torch.zeros((n, dim), dtype=torch.float64, device=DEV)
    for s in range(0, int(idx.numel()), 1 << 19):
        e = slice(s, s + (1 << 19))
        v = x[idx[e].long()].double() * (cf[idx[e].long()] * rf[dst[e]])[:, None]
        want.index_add_(0, dst[e], v)
        mag.index_add_(0, dst[e], v.abs())
    # weights off by a few eps, then a chain of at most 64 (chunk) + 32 (chunks) + 6 + 137 (segments) additions
    limit = 250 * 2.0 ** -24 * mag + (want.abs() * 2.0 ** -8 if dtype == torch.bfloat16 else 0) + 1e-30
    assert bool(((got.double() - want).abs() <= limit).all())


def test_the_least_entry_count_is_the_librarys():
    assert L.lib().fgl_aggregate_workspace_bytes(L.AGG_SEG_MIN_ENTRIES, 64, L.AGG_SUM, -1) > 0
    assert L.lib().fgl_aggregate_workspace_bytes(L.AGG_SEG_MIN_ENTRIES - 1, 64, L.AGG_SUM, -1) == 0
    assert L.lib().fgl_aggregate_workspace_bytes(L.AGG_SEG_MIN_ENTRIES, 64, L.AGG_EDGE, -1) == 0
    assert L.lib().fgl_aggregate_workspace_bytes(L.AGG_SEG_MIN_ENTRIES, 64, L.AGG_SUM, 128) == 0


@pytest.mark.parametrize("dim", [64, 300])
def test_the_mapping_names_the_second_pass(dim):
    ptr, idx, lens = _block(500)
    x = torch.zeros((500, dim), device=DEV)
    for kw, want in ((dict(mode="sum"), "segments"), (dict(mode="edge", edge_weight=torch.zeros((idx.numel(), 1), device=DEV)), "long_rows")):
        ops.aggregate(ptr, idx, x, zero_policy="zeros", **kw)
        assert L.lib().fgl_aggregate_last_mapping().decode().endswith(" + " + want)
