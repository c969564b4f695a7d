"""Degrees taken from row pointers (modes gcn_own / gcn_own_ptr) against the same sums with degree arrays -- the same numbers enter
the same formula, so bit for bit -- in every lane mapping; rows without entries cleared; a GCN layer with and without arrays."""
import pytest
import torch

import fastgl
from fastgl import ops

pytestmark = pytest.mark.gpu


def _csr(kind, gen, device):
    if kind == "fanout":
        lengths = torch.randint(0, 16, (3000,), generator=gen)
    elif kind == "few":
        lengths = torch.randint(0, 26, (150,), generator=gen)
    elif kind == "short":
        lengths = torch.randint(0, 3, (5000,), generator=gen)
    else:  # "hub": long rows among short ones
        lengths = torch.randint(0, 4, (2000,), generator=gen)
        lengths[7], lengths[900] = 1500, 200
    ptr = torch.zeros(len(lengths) + 1, dtype=torch.int64)
    ptr[1:] = torch.cumsum(lengths, 0)
    n_cols = 2 * len(lengths)
    idx = torch.randint(0, n_cols, (int(lengths.sum()),), generator=gen, dtype=torch.int32)
    return ptr.int().to(device), idx.to(device), len(lengths), n_cols


@pytest.mark.parametrize("dtype,dim", [(torch.float32, 20), (torch.float32, 100), (torch.float32, 602), (torch.bfloat16, 64), (torch.bfloat16, 33)])
@pytest.mark.parametrize("kind", ["fanout", "few", "short", "hub"])
def test_own_degrees_equal_degree_arrays(cuda, kind, dtype, dim):
    gen = torch.Generator().manual_seed(dim)
    ptr, idx, n, n_cols = _csr(kind, gen, cuda)
    x = torch.randn((n_cols, dim), generator=gen).to(cuda, dtype)
    row_deg = (ptr[1:] - ptr[:-1]).clamp(min=1)
    col_deg = torch.bincount(idx.long(), minlength=n_cols).int().clamp(min=1)
    col_ptr = torch.zeros(n_cols + 1, dtype=torch.int32, device=cuda)
    col_ptr[1:] = torch.cumsum(col_deg, 0)
    longest = 25 if kind == "few" else None
    want = fastgl.aggregate(ptr, idx, x, mode="gcn", row_norm=row_deg, col_norm=col_deg, zero_policy="self", longest_row=longest)
    for mode, col in (("gcn_own", col_deg), ("gcn_own_ptr", col_ptr)):
        got = fastgl.aggregate(ptr, idx, x, mode=mode, col_norm=col, zero_policy="self", longest_row=longest)
        assert torch.equal(got, want)
    cleared = ops.zero_empty_rows_(ptr, want.clone(), n)
    empty = ptr[1:] == ptr[:-1]
    assert torch.equal(cleared[~empty], want[~empty]) and not cleared[empty].any()


@pytest.mark.parametrize("order", ["gather_first", "product_first"])
def test_layer_without_degree_arrays(cuda, order):
    edge_ptr, edge_src = fastgl.graph.rmat_csr(20_000, 200_000, seed=3, device=cuda)
    sampler = fastgl.FusedMapSampler([5, 5], rng_seed=1, deterministic=True).set_graph(edge_ptr, edge_src)
    _, _, blocks = sampler.sample_blocks(None, torch.arange(600, dtype=torch.int32, device=cuda) * 31)
    for block in blocks:  # the inner one comes with its transposed form, the outer one without
        torch.manual_seed(2)
        x = torch.randn(block.num_src_nodes(), 40, device=cuda)
        layer = fastgl.GCNConv(40, 24, weight=True).to(cuda)
        layer.order = order
        g = torch.randn(block.num_dst_nodes(), 24, device=cuda)
        got = []
        for arrays in (True, False):
            xi = x.clone().requires_grad_()
            norms = (block.out_degrees().clamp(min=1), block.in_degrees().clamp(min=1)) if arrays else (None, None)
            y = layer(block.edge_ptr, block.src_local, norms[0], norms[1], block.num_dst_nodes(), xi, 5, block)
            layer.zero_grad()
            y.backward(g)
            got.append((y.detach(), xi.grad, layer.weights.grad.clone()))
        for a, b in zip(*got):
            assert torch.equal(a, b)
