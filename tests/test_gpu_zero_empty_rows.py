"""Rows without entries cleared in place: every width of store, rows at the edges of a wave's share of 16 or, of a million rows
and more, 64, strided rows; nothing else touched; and the look at many rows of which none is empty takes no longer than a launch."""
import pytest
import torch

from fastgl import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n, d, stride, offset", [
    (1, 1, 1, 0), (15, 4, 4, 0), (16, 100, 100, 0), (17, 256, 256, 0), (65, 3, 5, 1), (1000, 602, 602, 0), (4097, 8, 24, 8), (130, 1030, 1040, 2),
    (999_999, 4, 4, 0), (1_000_000, 4, 4, 0), (1_000_037, 3, 3, 0), (1_000_063, 7, 9, 1)])
def test_rows_without_entries_become_zeros(dtype, n, d, stride, offset):
    gen = torch.Generator().manual_seed(n * 7 + d)
    for share in (0.0, 0.4, 1.0):  # of rows without entries
        lengths = torch.where(torch.rand(n, generator=gen) < share, 0, torch.randint(1, 5, (n,), generator=gen))
        indptr = torch.cat([torch.zeros(1, dtype=torch.int64), lengths.cumsum(0)]).to(torch.int32)
        buf = torch.randn(n * stride + offset + 64, generator=gen).to(dtype)
        want = buf.clone()
        want.as_strided((n, d), (stride, 1), offset)[lengths == 0] = 0
        got = buf.cuda()
        ops.zero_empty_rows_(indptr.cuda(), got.as_strided((n, d), (stride, 1), offset), n)
        assert torch.equal(got.cpu(), want)


def test_a_look_at_many_rows(cuda):
    """Sixteen rows a wave made 2.4 M rows, none of them empty, twice a launch's time."""
    best = {}
    for n in (300_000, 2_400_000):
        indptr, x = torch.arange(n + 1, dtype=torch.int32, device=cuda), torch.zeros((n, 64), device=cuda)
        best[n] = float("inf")
        for _ in range(6):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            for _ in range(50):
                ops.zero_empty_rows_(indptr, x, n)
            end.record()
            end.synchronize()
            best[n] = min(best[n], begin.elapsed_time(end))
    assert best[2_400_000] < 1.5 * best[300_000]
