"""Long rows of large graphs, gathered class by class of their neighbours (csrc/fgl_aggregate.hip): rows around the limits of the long row, the row in classes and
the segment, in every mode, against float64; the sizes on either side of the rule; the same bits on every run."""
import pytest
import torch

from fastgl import _lib as L
from fastgl import ops

pytestmark = pytest.mark.gpu

LENGTHS = [0, 1, 127, 128, 129, 255, 256, 257, 300, 511, 512, 513, 1023, 1024, 1025, 4097, 9000, 85_000]


def _graph(cuda, n_rows, rest, seed):
    """The lengths above at both ends of the rows and `rest` entries in every other one; half of the neighbours are among a few hundred ids."""
    gen = torch.Generator(device=cuda).manual_seed(seed)
    lengths = torch.full((n_rows,), rest, dtype=torch.int64)
    lengths[:len(LENGTHS)] = torch.tensor(LENGTHS)
    lengths[-len(LENGTHS):] = torch.tensor(LENGTHS[::-1])
    ptr = torch.zeros(n_rows + 1, dtype=torch.int64)
    ptr[1:] = lengths.cumsum(0)
    n = int(ptr[-1])
    idx = torch.randint(0, n_rows, (n,), generator=gen, device=cuda)
    few = torch.randint(0, 300, (n,), generator=gen, device=cuda)
    idx = torch.where(torch.rand(n, generator=gen, device=cuda) < 0.5, few, idx).int()
    return ptr.int().to(cuda), idx, lengths


@pytest.mark.parametrize("n_rows,rest,D,dtype,classes", [
    (280_000, 46, 64, torch.float32, True), (260_000, 50, 65, torch.float32, True), (270_000, 47, 130, torch.float32, True), (280_000, 46, 602, torch.float32, True),
    (270_000, 48, 128, torch.bfloat16, True), (280_000, 40, 64, torch.float32, False), (280_000, 46, 60, torch.float32, False),
    (280_000, 46, 64, torch.bfloat16, False), (260_000, 50, 64, torch.float32, False)])
def test_against_float64(cuda, n_rows, rest, D, dtype, classes):
    print("classes", n_rows, rest, D, dtype, flush=True)
    ptr, idx, lengths = _graph(cuda, n_rows, rest, D)
    gen = torch.Generator(device=cuda).manual_seed(D + 1)
    x = torch.randn((n_rows, D), generator=gen, device=cuda).to(dtype)
    row_norm, col_norm = (torch.randint(1, 50, (n_rows,), generator=gen, device=cuda, dtype=torch.int32) for _ in range(2))
    rows = torch.cat((torch.arange(len(LENGTHS) + 5), torch.arange(n_rows - len(LENGTHS), n_rows)))
    first, n = ptr.cpu().long()[rows], lengths[rows]
    at = torch.cat([torch.arange(f, f + k) for f, k in zip(first.tolist(), n.tolist())]).to(cuda)  # the rows' entries
    which = torch.repeat_interleave(torch.arange(rows.numel()), n).to(cuda)
    n, rows, c = n.to(cuda), rows.to(cuda), idx[at].long()
    for mode in ("sum", "mean", "gcn", "colmean"):
        norms = dict(row_norm=row_norm if mode == "gcn" else None, col_norm=col_norm if mode in ("gcn", "colmean") else None)
        got = ops.aggregate(ptr, idx, x, mode=mode, zero_policy="zeros", **norms)
        assert (b"+ classes" in L.lib().fgl_aggregate_last_mapping()) == classes
        assert torch.equal(got, ops.aggregate(ptr, idx, x, mode=mode, zero_policy="zeros", **norms))
        w = torch.ones(at.numel(), dtype=torch.float64, device=cuda)
        if mode == "mean":
            w = 1 / n[which].double()
        elif mode == "gcn":
            w = (1 / col_norm[c].double()).sqrt() / row_norm[rows][which].double().sqrt()
        elif mode == "colmean":
            w = 1 / col_norm[c].double()
        terms = w[:, None] * x[c].double()
        want = torch.stack([t.sum(0) for t in terms.split(n.tolist())])
        size = torch.stack([t.abs().sum(0) for t in terms.split(n.tolist())])
        # a weight is three roundings, a term one, and a sum at most 64 in a chunk, n / 16 chunks, eight classes and n / 512 segments deep
        bound = (80 + n.double()[:, None] / 16) * 2.0 ** -24 * size + (want.abs() * 2.0 ** -8 if dtype == torch.bfloat16 else 0)
        assert bool(((got[rows].double() - want).abs() <= bound).all()), mode


def test_rows_of_a_larger_csr(cuda):
    """The C entry over a stretch of a CSR's rows, with the entries of that stretch as their bound: offsets that begin far beyond the scratch's ids."""
    lib, D, first = L.lib(), 64, 270_000
    ptr, idx, lengths = _graph(cuda, 2 * first, 48, 5)
    x = torch.randn((2 * first, D), generator=torch.Generator(device=cuda).manual_seed(6), device=cuda)
    rows, n = ptr[first:], int(ptr[-1] - ptr[first])
    assert n < int(ptr[first]) + 100_000 and n > 12_582_912
    out = torch.empty((first, D), device=cuda)
    ws_bytes = lib.fgl_aggregate_workspace_bytes_for(n, first, 2 * first, D, L.F32, L.AGG_SUM, -1)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=cuda)
    L.check(lib.fgl_aggregate_ws(rows.data_ptr(), idx.data_ptr(), first, None, x.data_ptr(), D, D, L.F32, L.AGG_SUM, L.ZERO_ZEROS, None, None, None, 1, None,
                                 -1, None, n, out.data_ptr(), D, ws.data_ptr(), ws_bytes, L.stream_handle()))
    assert b"+ classes" in lib.fgl_aggregate_last_mapping()
    for r in range(2 * first - len(LENGTHS), 2 * first):
        terms = x[idx[int(ptr[r]):int(ptr[r + 1])].long()].double()
        bound = (80 + lengths[r].item() / 16) * 2.0 ** -24 * terms.abs().sum(0)
        assert bool(((out[r - first].double() - terms.sum(0)).abs() <= bound).all())


def test_scratch_without_classes(cuda):
    """The workspace that fgl_aggregate_workspace_bytes asks for: segments, without classes; and a source of few rows, of which classes are not asked."""
    lib, D, n_rows = L.lib(), 64, 280_000
    ptr, idx, lengths = _graph(cuda, n_rows, 46, 7)
    n = int(ptr[-1])
    x = torch.randn((n_rows, D), generator=torch.Generator(device=cuda).manual_seed(8), device=cuda)
    out = torch.empty((n_rows, D), device=cuda)
    less, whole = lib.fgl_aggregate_workspace_bytes(n, D, L.AGG_SUM, -1), lib.fgl_aggregate_workspace_bytes_for(n, n_rows, n_rows, D, L.F32, L.AGG_SUM, -1)
    assert 0 < less < whole
    for ws_bytes, name in ((whole, b"+ classes + segments"), (whole - 1, b"+ segments"), (less, b"+ segments"), (less - 1, b"+ long_rows")):
        ws = torch.empty(ws_bytes, dtype=torch.uint8, device=cuda)
        L.check(lib.fgl_aggregate_ws(ptr.data_ptr(), idx.data_ptr(), n_rows, None, x.data_ptr(), D, D, L.F32, L.AGG_SUM, L.ZERO_ZEROS, None, None, None, 1, None,
                                     -1, None, n, out.data_ptr(), D, ws.data_ptr(), ws_bytes, L.stream_handle()))
        assert lib.fgl_aggregate_last_mapping().endswith(name) and (b"classes" in name or b"classes" not in lib.fgl_aggregate_last_mapping())
        for r in range(len(LENGTHS)):
            terms = x[idx[int(ptr[r]):int(ptr[r + 1])].long()].double()
            assert bool(((out[r].double() - terms.sum(0)).abs() <= (80 + lengths[r].item() / 16) * 2.0 ** -24 * terms.abs().sum(0)).all())
    few = ops.aggregate(ptr, idx % 300, x[:300], mode="sum", zero_policy="zeros")
    assert few.shape == (n_rows, D) and lib.fgl_aggregate_last_mapping().endswith(b"+ segments") and b"classes" not in lib.fgl_aggregate_last_mapping()
