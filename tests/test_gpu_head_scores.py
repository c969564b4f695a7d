"""fgl_head_scores (both score halves of a GAT layer in one pass) against float64 sums: head widths that are and are not whole
vectors, rows that do not fill a group of four, no destination rows and all of them."""
import pytest
import torch

import fastgl
from fastgl import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,width", [(1, 1), (1, 16), (4, 64), (4, 37), (3, 66), (8, 5), (2, 300), (1, 172), (1500, 2)])
@pytest.mark.parametrize("n,n_dst", [(1, 0), (1, 1), (3, 2), (4, 4), (1001, 250), (4099, 4097)])
def test_matches_float64(cuda, heads, width, n, n_dst):
    gen = torch.Generator(device=cuda).manual_seed(heads * 1000 + width + n)
    x = torch.randn((n, heads * width), generator=gen, device=cuda)
    al, ar = (torch.randn((1, heads, width), generator=gen, device=cuda) for _ in range(2))
    el, er = ops.head_scores(x, al, ar, n_dst)
    assert el.shape == (n, heads) and er.shape == (n_dst, heads)
    parts = x.double().view(n, heads, width)
    for got, a, rows in ((el, al, n), (er, ar, n_dst)):
        terms = parts[:rows] * a.double()
        # every lane adds width / 16 products and the lanes five more times: that many roundings of at most the sum of the magnitudes
        limit = (width / 16 + 6) * 2.0 ** -24 * terms.abs().sum(-1) + 1e-30
        assert ((got.double() - terms.sum(-1)).abs() <= limit).all()


def test_refuses_shapes_that_do_not_match(cuda):
    x, a = torch.zeros((5, 12), device=cuda), torch.zeros((1, 3, 4), device=cuda)
    with pytest.raises(RuntimeError):
        ops.head_scores(x, a, a, 6)
    with pytest.raises(RuntimeError):
        ops.head_scores(x[:, :8].contiguous(), a, a, 5)
    with pytest.raises(RuntimeError):
        ops.head_scores(x.cpu(), a, a, 5)


@pytest.mark.parametrize("grad", [False, True])
def test_layer_takes_any_leading_shape(cuda, grad):
    edge_ptr, edge_src = fastgl.graph.rmat_csr(2000, 20000, seed=3, device=cuda)
    sampler = fastgl.FusedMapSampler([5], rng_seed=1).set_graph(edge_ptr, edge_src)
    _, _, (block,) = sampler.sample_blocks(None, torch.arange(40, dtype=torch.int32, device=cuda) * 31)
    n = block.num_src_nodes()
    layer = fastgl.GATConv(12, 8, num_heads=2).to(cuda)
    x = torch.randn(n, 12, device=cuda)
    with torch.set_grad_enabled(grad):
        want = layer(block, x, 5)
        for shape in ((n, 1, 12), (1, n, 12)):
            assert torch.allclose(layer(block, x.view(shape), 5), want, rtol=1e-5, atol=1e-5)


def test_layer_takes_a_single_row_as_a_vector(cuda):
    block = fastgl.Block(torch.tensor([0, 1], dtype=torch.int32, device=cuda), torch.zeros(1, dtype=torch.int32, device=cuda), 1, 1)
    layer = fastgl.GATConv(12, 8, num_heads=2).to(cuda)
    x = torch.randn(12, device=cuda)
    assert torch.allclose(layer(block, x, 1), layer(block, x[None], 1), rtol=1e-5, atol=1e-5)
