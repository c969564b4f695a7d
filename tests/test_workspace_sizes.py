"""Sizes that the C ABI asks scratch of: no more than a launch of the same sizes and type would use."""
from fastgl import _lib as L


def test_weight_grad():
    lib = L.lib()
    # beyond what is formed in parts, which would want eight times as much (k = 100 K, 4096 x 4096: 64 x 64 tiles of one sum each)
    assert lib.fgl_weight_grad_workspace_bytes(100_000, 4096, 4096) < 70 << 20
    for k, m, n in ((3000, 602, 4000), (8000, 602, 1000), (107_000, 100, 256), (1000, 1000, 1000), (5, 64, 64)):
        fp32, bf16 = (lib.fgl_weight_grad_workspace_bytes_for(k, m, n, d) for d in (L.F32, L.BF16))
        assert bf16 <= fp32 == lib.fgl_weight_grad_workspace_bytes(k, m, n)
    assert 4 * lib.fgl_weight_grad_workspace_bytes_for(3000, 602, 4000, L.BF16) < lib.fgl_weight_grad_workspace_bytes_for(3000, 602, 4000, L.F32)


def test_aggregate():
    lib, n, nodes = L.lib(), 54_000_000, 2_400_000

    def size(D, dtype, rows=nodes, sources=nodes, longest=-1, entries=n):
        return lib.fgl_aggregate_workspace_bytes_for(entries, rows, sources, D, dtype, L.AGG_GCN, longest)

    plain = lib.fgl_aggregate_workspace_bytes(n, 64, L.AGG_GCN, -1)
    assert plain < 64 << 20 < size(64, L.F32)  # (a sum a segment; eight, and the ids)
    # rows of 128 bytes, few rows on either side, no row long enough: what is never gathered by classes asks for no more than the segments take
    assert plain == size(64, L.BF16) == size(64, L.F32, rows=8192) == size(64, L.F32, sources=8192) == size(64, L.F32, longest=256)
    assert size(64, L.F32, longest=257) > plain
    assert size(64, L.F32, sources=49_152) > plain == size(64, L.F32, sources=49_151)  # (12 MB of gathered rows)
    assert size(64, L.F32, longest=128) == 0 and size(64, L.F32, entries=1000) == 0
    assert size(3000, L.F32, entries=2_000_000_000) == lib.fgl_aggregate_workspace_bytes(2_000_000_000, 3000, L.AGG_GCN, -1)  # (classes would take more than 4 GiB)
