"""Products of the layers while something follows torch's operators: those stay torch's own then."""
import pytest
import torch
from torch.fx.experimental.proxy_tensor import make_fx
from torch.utils.flop_counter import FlopCounterMode

import fastgl
from fastgl import ops

pytestmark = pytest.mark.gpu


@pytest.fixture
def layer(cuda):
    torch.manual_seed(0)
    return fastgl.conv._Linear(20, 7).to(cuda)


def test_dispatch_modes_see_the_products(cuda, layer):
    x = torch.randn(33, 20, device=cuda)
    with torch.no_grad():
        graph = make_fx(lambda t: layer(t))(x)  # (real tensors under a dispatch mode)
        other = torch.randn(33, 20, device=cuda)
        assert torch.allclose(graph(other), torch.nn.functional.linear(other, layer.weight, layer.bias), rtol=1e-5, atol=1e-5)
    w = torch.randn(20, 7, device=cuda)
    with FlopCounterMode(display=False) as count:
        ops.row_product(x, w)
        ops.weight_grad(x, x[:, :5])
    assert count.get_total_flops() == 2 * 33 * 20 * 7 + 2 * 33 * 20 * 5
    x.requires_grad_()
    with FlopCounterMode(display=False) as count:
        layer(x).square().sum().backward()
    assert count.get_total_flops() == 3 * 2 * 33 * 20 * 7


def test_function_modes_see_the_layer(cuda, layer):
    seen = []

    class Mode(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    with Mode():
        layer(torch.randn(33, 20, device=cuda))
    assert torch.nn.functional.linear in seen


def test_a_default_device_follows_nothing(cuda):
    assert not ops._followed()
    with torch.device("cpu"):
        assert not ops._followed()
    with FlopCounterMode(display=False):
        assert ops._followed()


@pytest.mark.parametrize("grad", [False, True])
def test_compiled(cuda, layer, grad):
    x = torch.randn(33, 20, device=cuda)
    with torch.set_grad_enabled(grad):
        got = torch.compile(layer, fullgraph=True, backend="eager")(x)
        assert torch.allclose(got, torch.nn.functional.linear(x, layer.weight, layer.bias), rtol=1e-5, atol=1e-5)


def test_batched_gradients_of_the_layer(cuda, layer):
    x = torch.randn(6, 20, device=cuda, requires_grad=True)
    y = layer(x)
    v = torch.eye(42, device=cuda).view(42, 6, 7)
    got = torch.autograd.grad(y, (x, layer.weight, layer.bias), v, is_grads_batched=True)
    want = torch.autograd.grad(torch.nn.functional.linear(x, layer.weight, layer.bias), (x, layer.weight, layer.bias), v, is_grads_batched=True)
    for a, b in zip(got, want):
        assert torch.allclose(a, b, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("kind", ["gcn", "gin"])
def test_batched_gradients_of_a_first_layer(cuda, kind):
    edge_ptr, edge_src = fastgl.graph.rmat_csr(2000, 20000, seed=3, device=cuda)
    sampler = fastgl.FusedMapSampler([3], rng_seed=1).set_graph(edge_ptr, edge_src)
    _, _, (block,) = sampler.sample_blocks(None, torch.arange(5, dtype=torch.int32, device=cuda) * 31)
    x = torch.randn(block.num_src_nodes(), 8, device=cuda)
    if kind == "gcn":
        layer = fastgl.GCNConv(8, 3, weight=True).to(cuda)
        layer.order = "gather_first"
        y = layer(block.edge_ptr, block.src_local, None, None, block.num_dst_nodes(), x, 3, block)
    else:
        layer = fastgl.GINConv(8, 3, weight=True).to(cuda)
        y = layer(block.edge_ptr, block.src_local, block.num_dst_nodes(), x, 3, block)
    v = torch.eye(y.numel(), device=cuda).view(-1, *y.shape)
    (got,) = torch.autograd.grad(y, (layer.weights,), v, is_grads_batched=True, retain_graph=True)
    for i in (0, y.numel() - 1):
        (want,) = torch.autograd.grad(y, (layer.weights,), v[i], retain_graph=True)
        assert torch.allclose(got[i], want, rtol=1e-5, atol=1e-5)
