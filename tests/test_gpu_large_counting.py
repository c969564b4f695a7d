"""cal_deg and block_transpose where they change form (counted with atomics, in LDS ranges, or partitioned into buckets first), hub ids, ids outside the range, rows of every length and gaps of empty rows.  Whole
numbers throughout: equal to torch.bincount, and to the stable sort by column where order is promised or sorted away."""
import pytest
import torch

import fastgl
from fastgl import _lib as L

pytestmark = pytest.mark.gpu

M = 1 << 20


def _ids(n, bins, gen, device, hub):
    ids = torch.randint(0, bins, (n,), generator=gen, device=device, dtype=torch.int32)
    if hub:  # a third of the mentions to one id, and a few that are no ids at all
        ids[torch.rand(n, generator=gen, device=device) < 0.33] = bins // 2
        ids[::1001] = -1
        ids[5::1003] = bins + 7
    return ids


@pytest.mark.parametrize("hub", [False, True])
@pytest.mark.parametrize("n,bins", [((1 << 16) - 1, 1000), (1 << 16, 1 << 15), (1 << 16, (1 << 15) + 1), ((1 << 18) - 1, 1000), (1 << 18, 16384), ((1 << 18) + 3, 16385), (M + 5, 1 << 19), (M, (1 << 19) + 1),
                                    (300_001, 1), (4 * M - 1, 300_000), (4 * M, 1), (4 * M, 2048), (4 * M + 8191, 2049),
                                    (5 * M + 77, 3_000_001), (4 * M, 5 * M), (M, 8 * M + 9)])
def test_cal_deg(cuda, n, bins, hub):
    gen = torch.Generator(device=cuda).manual_seed(n + bins)
    ids = _ids(n, bins, gen, cuda, hub)
    got = fastgl.cal_deg(ids, bins)
    valid = ids[(ids >= 0) & (ids < bins)].long()
    assert torch.equal(got.long(), torch.bincount(valid, minlength=bins))


@pytest.mark.parametrize("n_max,n,bins", [(1 << 16, 60_000, 1 << 15), (1 << 18, 5, 16385), (1 << 18, 0, 1000), (4 * M, M + 1, 300_000), (4 * M, 0, 2048)])
def test_cal_deg_of_a_count_on_the_device(cuda, n_max, n, bins):
    gen = torch.Generator(device=cuda).manual_seed(n_max + n)
    ids = _ids(n_max, bins, gen, cuda, False)
    lib = fastgl.lib()
    d_n = torch.tensor([n], dtype=torch.int32, device=cuda)
    got = torch.full((bins,), -7, dtype=torch.int32, device=cuda)
    ws = L.workspace(lib.fgl_cal_deg_workspace_bytes(n_max, bins), cuda)
    L.check(lib.fgl_cal_deg_ws(L.ptr(ids), n_max, L.ptr(d_n), L.ptr(got), bins, L.ptr(ws), ws.numel(), L.stream_handle()))
    assert torch.equal(got.long(), torch.bincount(ids[:n].long(), minlength=bins))


@pytest.mark.parametrize("n", [(1 << 16) - 1, 1 << 16, 1 << 18, 4 * M])
def test_cal_deg_into_no_bins(cuda, n):
    assert fastgl.cal_deg(torch.zeros(n, dtype=torch.int32, device=cuda), 0).shape == (0,)


def _csr(lengths, device):
    ptr = torch.zeros(len(lengths) + 1, dtype=torch.int64)
    ptr[1:] = torch.cumsum(lengths, 0)
    return ptr.int().to(device)


def _lengths(kind, gen):
    if kind == "fanout":      # rows of a sampled block
        return torch.randint(0, 26, (20_000,), generator=gen)
    if kind == "hub":         # one row of 100 K entries among short and empty ones
        x = torch.randint(0, 4, (30_000,), generator=gen)
        x[17] = 100_000
        return x
    if kind == "gaps":        # long gaps of empty rows, also in front and at the end
        x = torch.zeros(200_000, dtype=torch.int64)
        x[100_000:100_040] = 701
        x[199_000] = 3
        return x
    if kind == "large":       # past the partition's threshold, hub rows and a gap
        x = torch.randint(0, 15, (600_000,), generator=gen)
        x[5] = 300_000
        x[400_000:520_000] = 0
        x[599_000] = 50_001
        return x
    return torch.tensor([1])  # "one"


@pytest.mark.parametrize("edge_ids", [False, True])
@pytest.mark.parametrize("kind,n_cols", [("one", 1), ("fanout", 3000), ("hub", 70_000), ("gaps", 500), ("large", 1), ("large", 2_500_000),
                                         ("large", 4096), ("large", 8 * M + 9),  # (buckets of 2^13 columns)
                                         ("large", 16 * M + 5)])                 # (too wide for buckets: eight counters a column)
def test_block_transpose(cuda, kind, n_cols, edge_ids):
    gen = torch.Generator().manual_seed(n_cols)
    lengths = _lengths(kind, gen)
    ptr = _csr(lengths, cuda)
    nnz = int(lengths.sum())
    cols = torch.randint(0, n_cols, (nnz,), generator=gen, dtype=torch.int32)
    cols[torch.rand(nnz, generator=gen) < 0.1] = n_cols // 3  # a hub column
    cols = cols.to(cuda)
    n_rows = len(lengths)
    got = fastgl.block_transpose(ptr, cols, n_rows, n_cols, edge_ids=edge_ids)
    rows = torch.repeat_interleave(torch.arange(n_rows, device=cuda), lengths.to(cuda))
    counts = torch.bincount(cols.long(), minlength=n_cols)
    want_ptr = torch.zeros(n_cols + 1, dtype=torch.int64, device=cuda)
    want_ptr[1:] = torch.cumsum(counts, 0)
    assert torch.equal(got[0].long(), want_ptr)
    longest = int(counts.max())
    assert int(got[0].fgl_longest_row) == longest if longest > 32 else int(got[0].fgl_longest_row) <= 32
    # the order inside a column is not promised: compare (column, row[, entry]) after sorting
    col_of = torch.repeat_interleave(torch.arange(n_cols, device=cuda), counts)
    assert torch.equal(torch.sort(col_of * n_rows + got[1].long()).values, torch.sort(cols.long() * n_rows + rows).values)
    if edge_ids:
        e = got[2].long()
        assert torch.equal(torch.sort(e).values, torch.arange(nnz, device=cuda))
        assert torch.equal(cols.long()[e], col_of) and torch.equal(rows[e], got[1].long())


@pytest.mark.parametrize("sorted_rows", [False, True])
@pytest.mark.parametrize("first,lengths,n_cols", [
    (1, [3, 0, 2], 4), (1023, [1], 5), (5000, [3, 0, 4000, 3000], 900),  # tiles of 1024 entries, one by one
    (9000, [40_000, 0, 230_000], 3000), (300_000, [1] * 9, 70_000)])     # tiles of 8192, through the buckets
def test_block_transpose_of_a_slice(cuda, first, lengths, n_cols, sorted_rows):
    """Offsets that do not start at zero: the entries in front count as row 0's, whatever the form."""
    print("slice from", first, lengths, n_cols, sorted_rows, flush=True)
    lens = torch.tensor(lengths)
    ptr = _csr(lens, cuda) + first
    nnz = first + int(lens.sum())
    cols = torch.randint(0, n_cols, (nnz,), generator=torch.Generator().manual_seed(first), dtype=torch.int32).to(cuda)
    t_ptr, t_idx, t_edge = fastgl.block_transpose(ptr, cols, len(lengths), n_cols, edge_ids=True, sorted_rows=sorted_rows)
    lens[0] += first
    rows = torch.repeat_interleave(torch.arange(len(lengths)), lens).to(cuda)
    counts = torch.bincount(cols.long(), minlength=n_cols)
    assert torch.equal(t_ptr[1:].long(), torch.cumsum(counts, 0)) and int(t_ptr[0]) == 0
    e = t_edge.long()
    assert torch.equal(torch.sort(e).values, torch.arange(nnz, device=cuda))
    assert torch.equal(cols.long()[e], torch.repeat_interleave(torch.arange(n_cols, device=cuda), counts)) and torch.equal(rows[e], t_idx.long())


@pytest.mark.parametrize("rows,cols,nnz_max", [(5000, 3000, M), (4999, 1, M + 7), (0, 3000, M), (5000, 3000, M - 1)])
def test_block_transpose_of_sizes_on_the_device(cuda, rows, cols, nnz_max):
    """A block whose sizes the host knows bounds of only: from 2^20 entries on with eight counters a column, below with one."""
    print("device sizes", rows, cols, nnz_max, flush=True)
    gen = torch.Generator().manual_seed(rows + nnz_max)
    rows_max, cols_max = 6000, 4000
    lens = torch.randint(0, 300, (rows,), generator=gen)
    if rows:
        lens[rows // 2] = 50_000  # a hub
    ptr = torch.full((rows_max + 1,), -1, dtype=torch.int32, device=cuda)  # (past the actual rows: never read)
    ptr[:rows + 1] = _csr(lens, cuda)
    nnz = int(lens.sum())
    assert nnz <= nnz_max
    idx = torch.full((nnz_max,), -1, dtype=torch.int32)
    idx[:nnz] = torch.randint(0, cols, (nnz,), generator=gen, dtype=torch.int32)
    idx[:nnz][torch.rand(nnz, generator=gen) < 0.1] = cols // 3
    idx = idx.to(cuda)
    d_rows, d_cols = (torch.tensor([v], dtype=torch.int32, device=cuda) for v in (rows, cols))
    t_ptr = torch.full((cols_max + 1,), -7, dtype=torch.int32, device=cuda)
    t_idx, t_edge = (torch.full((nnz_max,), -7, dtype=torch.int32, device=cuda) for _ in range(2))
    longest = torch.full((1,), -7, dtype=torch.int32, device=cuda)
    lib = fastgl.lib()
    ws = L.workspace(lib.fgl_block_transpose_workspace_bytes(cols_max, nnz_max, 0), cuda)
    L.check(lib.fgl_block_transpose(L.ptr(ptr), L.ptr(idx), rows_max, L.ptr(d_rows), cols_max, L.ptr(d_cols), nnz_max, L.ptr(t_ptr), L.ptr(t_idx),
                                    L.ptr(t_edge), L.ptr(longest), 0, L.ptr(ws), ws.numel(), L.stream_handle()))
    of_row = torch.repeat_interleave(torch.arange(rows), lens).to(cuda)
    counts = torch.bincount(idx[:nnz].long(), minlength=cols)
    assert int(t_ptr[0]) == 0 and torch.equal(t_ptr[1:cols + 1].long(), torch.cumsum(counts, 0))
    top = int(counts.max())
    assert int(longest) == top if top > 32 else int(longest) <= 32
    e = t_edge[:nnz].long()
    assert torch.equal(torch.sort(e).values, torch.arange(nnz, device=cuda))
    assert torch.equal(idx[:nnz].long()[e], torch.repeat_interleave(torch.arange(cols, device=cuda), counts))
    assert torch.equal(of_row[e], t_idx[:nnz].long())
    assert bool((t_idx[nnz:] == -7).all()) and bool((t_edge[nnz:] == -7).all())
