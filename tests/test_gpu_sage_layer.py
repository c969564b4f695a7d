"""A GraphSAGE layer formed as a whole against the same layer part by part (which a hook on one of its parts makes it), and the two kernels'
forms behind it against float64: two pairs of operands, sums added to what is there, sizes at the edges of tiles and steps."""
import numpy as np
import pytest
import torch

import fastgl
from fastgl import ops

pytestmark = pytest.mark.gpu


# two operands' k around a step (8 / 16), m around a tile (32, 64, 128), n around a vector and a tile
@pytest.mark.parametrize("dtype,rel", [(torch.float32, 1e-6), (torch.bfloat16, 6e-3)])  # (bf16: two values and their sum rounded, 2^-9 each)
@pytest.mark.parametrize("m,k0,k1,n", [(1, 2, 2, 1), (33, 8, 16, 32), (64, 34, 2, 66), (127, 100, 256, 47), (200, 16, 130, 128), (1025, 64, 62, 256),
                                       (70_000, 32, 48, 96), (65_537, 60, 70, 256), (65_537, 64, 62, 256), (131_009, 258, 254, 64)])
def test_two_products_in_one_pass(cuda, dtype, rel, m, k0, k1, n):
    print("pair", dtype, m, k0, k1, n, flush=True)
    gen = torch.Generator().manual_seed(m + n)
    x, h, ws, wn, bias = (torch.randn(s, generator=gen).to(dtype) for s in ((m, k0), (m, k1), (n, k0), (n, k1), (n,)))
    dev = [t.to(cuda) for t in (x, ws, h, wn, bias)]
    with torch.no_grad():
        got = ops.row_product_sum(*dev)
        want = x.double() @ ws.double().t() + h.double() @ wn.double().t() + bias.double()
        assert float((got.cpu().double() - want).norm() / want.norm()) < rel
        apart = ops.row_product(dev[0], dev[1], transposed=True) + ops.row_product(dev[2], dev[3], transposed=True, bias=dev[4])
        assert dtype == torch.float32 or torch.equal(got, apart)  # (the same sums, rounded at the same places)
        g = torch.randn((m, n), generator=gen).to(dtype)
        base = torch.randn((m + 3, k0), generator=gen).to(dtype)
        got = ops.row_product_add_(base.to(cuda), g.to(cuda), dev[1])
        want = base.double()
        want[:m] += g.double() @ ws.double()
        assert torch.equal(got[m:].cpu(), base[m:])
        apart = base.to(cuda)
        apart[:m] += ops.row_product(g.to(cuda), dev[1])
        assert dtype == torch.float32 or torch.equal(got, apart)
        assert float((got.cpu().double() - want).norm() / want.norm()) < rel


# wide vectors need a thousand waves; rows that are no whole number of them, whose last vector lies across two tiles (129, 514) or two lanes
@pytest.mark.parametrize("dtype,rel", [(torch.float32, 1e-6), (torch.bfloat16, 6e-3)])
@pytest.mark.parametrize("m,k,n", [(12_000, 8, 129), (9_000, 8, 514), (9_000, 16, 130), (12_000, 8, 98), (12_000, 8, 256)])
def test_sums_are_added_once(cuda, dtype, rel, m, k, n):
    print("add", dtype, m, k, n, flush=True)
    gen = torch.Generator().manual_seed(n)
    a, b, base = (torch.randn(s, generator=gen).to(dtype) for s in ((m, k), (k, n), (m + 1, n)))
    with torch.no_grad():
        got = ops.row_product_add_(base.to(cuda), a.to(cuda), b.to(cuda)).cpu().double()
    want = base.double()
    want[:m] += a.double() @ b.double()
    assert float(((got - want).norm(dim=0) / want.norm(dim=0)).max()) < rel  # (column by column: a sum of one column added twice is seen)


def _setup(cuda, dtype, dim, hidden, classes):
    edge_ptr, edge_src = fastgl.graph.rmat_csr(20_000, 200_000, seed=3, device=cuda)
    sampler = fastgl.FusedMapSampler([10, 8], rng_seed=1, deterministic=True).set_graph(edge_ptr, edge_src)
    seeds = torch.arange(0, 20_000, 37, device=cuda).int()
    nodes, _, blocks = sampler.sample_blocks(None, seeds)
    torch.manual_seed(0)
    model = fastgl.SAGE(dim, hidden, classes, 2).to(cuda).to(dtype)
    feat = torch.randn((20_000, dim), device=cuda).to(dtype)
    return model, nodes, blocks, feat


def _step(model, nodes, blocks, feat, from_table, hooked, grad_of_input=False, frozen=()):
    handles = [layer.fc_self.register_forward_hook(lambda *a: None) for layer in model.layers] if hooked else []
    for name, p in model.named_parameters():
        p.requires_grad_(name not in frozen)
        p.grad = None
    x = feat if from_table else feat[nodes.long()]
    x = x.detach().clone().requires_grad_(grad_of_input)
    out = model(blocks, x, input_nodes=nodes if from_table else None)
    (out.float() ** 2).mean().backward()
    for h in handles:
        h.remove()
    return [out.detach()] + [p.grad for p in model.parameters()] + [x.grad]


@pytest.mark.parametrize("dtype,rel", [(torch.float32, 2e-6), (torch.bfloat16, 1e-5)])  # (bf16: the same sums, rounded at the same places)
@pytest.mark.parametrize("dim,hidden,classes", [(32, 64, 16), (100, 48, 47), (2, 2, 1)])
@pytest.mark.parametrize("from_table,grad_of_input", [(False, False), (False, True), (True, False), (True, True)])
def test_whole_layers_are_their_parts(cuda, dtype, rel, dim, hidden, classes, from_table, grad_of_input):
    print("sage", dtype, dim, hidden, classes, from_table, grad_of_input, flush=True)
    args = _setup(cuda, dtype, dim, hidden, classes)
    for frozen in ((), ("layers.0.fc_neigh.weight", "layers.1.fc_neigh.bias"), ("layers.0.fc_self.weight", "layers.1.fc_self.weight", "layers.0.fc_neigh.bias")):
        whole = _step(*args, from_table, False, grad_of_input, frozen)
        parts = _step(*args, from_table, True, grad_of_input, frozen)
        for a, b in zip(whole, parts):
            assert (a is None) == (b is None)
            if a is not None and float(b.float().norm()) > 0:
                assert float((a.double() - b.double()).norm() / b.double().norm()) < rel
    with torch.no_grad():
        model, nodes, blocks, feat = args
        x = (feat, nodes) if from_table else (feat[nodes.long()], None)
        assert torch.equal(model(blocks, *x), whole[0])


def test_what_calls_the_parts_still_does(cuda):
    """Hooks, replaced parts, modes, autocast, saved-tensor hooks and forward-mode differentiation see what they saw."""
    from torch.utils.flop_counter import FlopCounterMode
    model, nodes, blocks, feat = _setup(cuda, torch.float32, 32, 16, 8)
    x = feat[nodes.long()]
    calls = []
    handle = torch.nn.modules.module.register_module_forward_hook(lambda m, i, o: calls.append(type(m).__name__))
    model(blocks, x)
    handle.remove()
    assert calls.count("_Linear") == 4
    with FlopCounterMode(display=False) as flops:
        model(blocks, x)
    assert flops.get_total_flops() >= sum(2 * 2 * b.num_dst_nodes() * d * o for b, (d, o) in zip(blocks, ((32, 16), (16, 8))))
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert model.layers[0](blocks[0], x).dtype == torch.bfloat16
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t, lambda t: t):
        model(blocks, x).sum().backward()
    assert len(packed) >= 8
    whole = model(blocks, x)
    model.layers[0].fc_self = torch.nn.Sequential(model.layers[0].fc_self)
    assert torch.allclose(model(blocks, x), whole, rtol=1e-4, atol=1e-5)


def test_layers_whose_own_rows_are_not_one_for_each_destination(cuda):
    """One row that stands for all destinations is repeated, and its gradient summed; other numbers of rows are refused."""
    model, nodes, blocks, feat = _setup(cuda, torch.float32, 32, 16, 8)
    layer, block, x = model.layers[0], blocks[0], feat[nodes.long()]
    def step(hooked):
        handle = layer.fc_self.register_forward_hook(lambda *a: None) if hooked else None
        one = x[:1].clone().requires_grad_()
        out = layer(block, x, feat_dst=one)
        grads = torch.autograd.grad((out ** 2).mean(), [one] + list(layer.parameters()))
        if handle is not None:
            handle.remove()
        return [out.detach()] + list(grads)
    for a, b in zip(step(False), step(True)):
        assert a.shape == b.shape and float((a - b).norm() / b.norm()) < 2e-6
    with pytest.raises(RuntimeError):
        layer(block, x, feat_dst=x[:2])
    # (two destinations of one source, whose only row stands for both)
    ptr, ids = torch.tensor([0, 1, 2], dtype=torch.int32, device=cuda), torch.zeros(2, dtype=torch.int32, device=cuda)
    few = fastgl.Block(ptr, ids, 1, 2)
    one = x[:1].clone().requires_grad_()
    out = layer(few, one)
    got, = torch.autograd.grad(out.sum(), one)
    want = 2 * (layer.fc_self.weight + layer.fc_neigh.weight).detach().sum(0)
    assert out.shape == (2, 16) and float((got[0] - want).norm() / want.norm()) < 2e-6
    with pytest.raises(RuntimeError):
        ops.row_product_add_(torch.zeros((1, 32), device=cuda), torch.zeros((2, 16), device=cuda), layer.fc_self.weight.detach())


def test_gradients_of_gradients_of_the_weights(cuda):
    model, nodes, blocks, feat = _setup(cuda, torch.float32, 16, 8, 4)
    x, layer = feat[nodes.long()], model.layers[0]
    def penalty(hooked):
        handle = layer.fc_self.register_forward_hook(lambda *a: None) if hooked else None
        out = layer(blocks[0], x)
        g = torch.autograd.grad((out ** 3).sum(), list(layer.parameters()), create_graph=True)
        second = torch.autograd.grad(sum((t ** 2).sum() for t in g), list(layer.parameters()))
        if handle is not None:
            handle.remove()
        return second
    for a, b in zip(penalty(False), penalty(True)):
        assert float((a - b).norm() / b.norm()) < 1e-5


@pytest.mark.parametrize("own_rows", [True, False])
def test_gradients_of_gradients_reach_what_lies_below(cuda, own_rows):
    """A penalty on the second layer's weight gradients, differentiated by the input and by every weight, the first layer's among them."""
    model, nodes, blocks, feat = _setup(cuda, torch.float32, 16, 8, 4)
    x = feat[nodes.long()].requires_grad_()
    params = list(model.parameters())
    def penalty(hooked):
        handles = [layer.fc_self.register_forward_hook(lambda *a: None) for layer in model.layers] if hooked else []
        h = model.layers[0](blocks[0], x)
        out = model.layers[1](blocks[1], h) if own_rows else model.layers[1](blocks[1], h, feat_dst=h[:blocks[1].num_dst_nodes()] * 2)
        g = torch.autograd.grad((out ** 3).sum(), list(model.layers[1].parameters()), create_graph=True)
        second = torch.autograd.grad(sum((t ** 2).sum() for t in g), [x] + params)
        for handle in handles:
            handle.remove()
        return second
    for a, b in zip(penalty(False), penalty(True)):
        assert float(b.norm()) > 0 and float((a - b).norm() / b.norm()) < 1e-5


def test_what_is_saved_is_what_the_products_save(cuda):
    """Saved-tensor hooks see the inputs of the products, of as many rows, and rows that only the aggregation reads may change in place."""
    model, nodes, blocks, feat = _setup(cuda, torch.float32, 16, 8, 4)
    layer, block = model.layers[0], blocks[0]
    x, n_dst = feat[nodes.long()].requires_grad_(), block.num_dst_nodes()
    def saved(hooked):
        shapes = []
        handle = layer.fc_self.register_forward_hook(lambda *a: None) if hooked else None
        with torch.autograd.graph.saved_tensors_hooks(lambda t: shapes.append(tuple(t.shape)) or t, lambda t: t):
            layer(block, x).sum().backward()
        if handle is not None:
            handle.remove()
        return sorted(shapes)
    assert saved(False) == saved(True) and saved(False).count((n_dst, 16)) == 2
    src, own = (t.detach().clone().requires_grad_() for t in (x, x[:n_dst]))
    with torch.no_grad():
        want = layer(block, src, feat_dst=own)
    out = layer(block, src, feat_dst=own)
    with torch.no_grad():
        src.zero_()
    out.sum().backward()
    assert torch.equal(out.detach(), want) or torch.allclose(out, want, rtol=1e-5, atol=1e-5)
    assert src.grad.shape == src.shape and own.grad.shape == own.shape
