"""The partition behind large counts and transposes, at the edges of what it puts in order in LDS: tiles of 8192 entries, segments of
8192 to 32768, buckets of 2^11 to 2^13 columns, entries stored in order or as they are met; sorted ids (runs of equal ones), ids in a band, ids that
start on any word, and ids that are none.
Whole numbers, equal to torch.bincount and to the sorted pairs."""
import pytest
import torch

import fastgl

pytestmark = pytest.mark.gpu

M = 1 << 20


def _ids(kind, n, bins, gen, device):
    if kind == "sorted":
        return (torch.arange(n, device=device) * bins // max(n, 1)).int()
    if kind == "band":
        at = torch.arange(n, device=device) * bins // max(n, 1) + torch.randint(0, 64, (n,), generator=gen, device=device)
        return at.clamp(max=bins - 1).int()
    ids = torch.randint(0, bins, (n,), generator=gen, device=device, dtype=torch.int32)
    if kind == "runs":  # runs of 1..40 equal ids, none of them at the same place in a lane's sixteen
        ids = torch.repeat_interleave(ids, torch.randint(1, 41, (n,), generator=gen, device=device))[:n].contiguous()
    if kind == "hub":
        ids[torch.rand(n, generator=gen, device=device) < 0.4] = bins - 1
        ids[::997] = -1
        ids[3::991] = bins
    return ids


@pytest.mark.parametrize("kind", ["sorted", "runs", "hub"])
@pytest.mark.parametrize("n,bins,first", [(4 * M, 2048, 0), (4 * M + 1, 2049, 1), (4 * M + 8191, 600_000, 3), (4 * M + 8192, 4096, 2),
                                          (4 * M + 8193, 5 * M, 1), (M + 32767, M, 0), (M + 32769, M, 1)])
def test_counts(cuda, kind, n, bins, first):
    print("counts", kind, n, bins, first, flush=True)
    gen = torch.Generator(device=cuda).manual_seed(n)
    ids = _ids(kind, n + first, bins, gen, cuda)[first:]
    ok = ids[(ids >= 0) & (ids < bins)].long()
    assert torch.equal(fastgl.cal_deg(ids, bins).long(), torch.bincount(ok, minlength=bins))


@pytest.mark.parametrize("edge_ids", [False, True])
@pytest.mark.parametrize("kind", ["sorted", "runs", "hub", "band"])
@pytest.mark.parametrize("n,cols", [((1 << 18), 2048), ((1 << 18) + 1, 2049), (32 * 8192 + 8191, 4 * M + 1), (300_000, 1), (M + 8193, 100_000),
                                    ((1 << 18) + 1, 9 * M), (2 * M, 127 * 2048), (2 * M, 128 * 2048), (2 * M + 1, 300_000), (6 * M, 5 * M), (4 * M, 2047)])
def test_transposes(cuda, kind, n, cols, edge_ids):
    print("transposes", kind, n, cols, edge_ids, flush=True)
    gen = torch.Generator(device=cuda).manual_seed(n + cols)
    ids = _ids("runs" if kind == "hub" and cols == 1 else kind, n, cols, gen, cuda).clamp(0, cols - 1)
    n_rows = n // 7 + 1
    ptr = (torch.arange(n_rows + 1, device=cuda) * 7).clamp(max=n).int()
    got = fastgl.block_transpose(ptr, ids, n_rows, cols, edge_ids=edge_ids)
    counts = torch.bincount(ids.long(), minlength=cols)
    assert torch.equal(got[0][1:].long(), torch.cumsum(counts, 0)) and int(got[0][0]) == 0
    col_of = torch.repeat_interleave(torch.arange(cols, device=cuda), counts)
    rows = torch.arange(n, device=cuda) // 7
    assert torch.equal(torch.sort(col_of * n_rows + got[1].long()).values, torch.sort(ids.long() * n_rows + rows).values)
    if edge_ids:
        e = got[2].long()
        assert torch.equal(torch.sort(e).values, torch.arange(n, device=cuda)) and torch.equal(ids.long()[e], col_of)
        assert torch.equal(rows[e], got[1].long())
