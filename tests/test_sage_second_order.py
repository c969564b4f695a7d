"""Gradients of gradients through GraphSAGE layers formed as a whole, on the CPU: the device operators behind the layer are replaced by
torch's in float64, and every second derivative is compared with the one of the same layers written in plain torch."""
import pytest
import torch

from fastgl import conv, ops
from fastgl.sampler import Block


def _dense(ptr, idx, n_src):
    lens = (ptr[1:] - ptr[:-1]).long()
    a = torch.zeros((lens.numel(), n_src), dtype=torch.float64)
    rows = torch.repeat_interleave(torch.arange(lens.numel()), lens)
    a.index_put_((rows, idx.long()), torch.ones(idx.numel(), dtype=torch.float64), accumulate=True)
    return a, lens.clamp(min=1).double()


@pytest.fixture
def operators(monkeypatch):
    def aggregate(indptr, indices, feat, mode, zero_policy, n_rows, col_norm=None):
        a, lens = _dense(indptr, indices, feat.size(0))
        a = a / lens[:, None] if mode == "mean" else a / (col_norm[1:] - col_norm[:-1]).clamp(min=1).double()[None, :]
        return (a @ feat).detach()  # (the operator records nothing)
    def row_product(a, b, transposed=False, bias=None):
        out = a @ (b.t() if transposed else b)
        return out if bias is None else out + bias
    def weight_grad(a, b, column_sums=False):
        return (a.t() @ b, a.sum(0)) if column_sums else a.t() @ b
    def row_product_add_(out, a, b):
        out[:a.size(0)] += a @ b
        return out
    for name, f in dict(aggregate=aggregate, row_product=row_product, weight_grad=weight_grad, row_product_add_=row_product_add_,
                        row_product_sum=lambda *a: None).items():
        monkeypatch.setattr(ops, name, f)


def _block(n_src, n_dst, gen):
    lens = torch.randint(0, 4, (n_dst,), generator=gen)
    ptr = torch.zeros(n_dst + 1, dtype=torch.int32)
    ptr[1:] = torch.cumsum(lens, 0)
    idx = torch.randint(0, n_src, (int(ptr[-1]),), generator=gen, dtype=torch.int32)
    order = torch.argsort(idx, stable=True)
    t_ptr = torch.zeros(n_src + 1, dtype=torch.int32)
    t_ptr[1:] = torch.cumsum(torch.bincount(idx.long(), minlength=n_src), 0)
    block = Block(ptr, idx, n_src, n_dst)
    block._transposed = (t_ptr, torch.repeat_interleave(torch.arange(n_dst), lens)[order].int(), order.int())
    return block


def _plain(block, x, own, w_self, w_neigh, bias):
    a, lens = _dense(block.edge_ptr, block.src_local, x.size(0))
    return own @ w_self.t() + (a / lens[:, None]) @ x @ w_neigh.t() + bias


@pytest.mark.parametrize("wanted", ["input", "first layer", "all"])
@pytest.mark.parametrize("constant_gradient", [False, True])
def test_penalty_on_the_gradients_of_the_weights(operators, wanted, constant_gradient):
    gen = torch.Generator().manual_seed(3)
    blocks = [_block(30, 17, gen), _block(17, 8, gen)]
    rand = lambda *s: torch.randn(s, generator=gen, dtype=torch.float64).requires_grad_()
    first, second = (rand(6, 5), rand(6, 5), rand(6)), (rand(3, 6), rand(3, 6), rand(3))
    x = rand(30, 5)
    weigh = torch.randn((8, 3), generator=gen, dtype=torch.float64)
    to = {"input": [x], "first layer": list(first), "all": [x, *first, *second]}[wanted]

    def second_order(layer):
        out = layer(blocks[1], layer(blocks[0], x, first), second)
        # (a gradient of the output that does not depend on it: all of the second derivative comes through what the products saved)
        loss = (out * weigh).sum() if constant_gradient else (out ** 3).sum()
        g = torch.autograd.grad(loss, second, create_graph=True)
        return torch.autograd.grad(sum((t ** 2).sum() for t in g), to, allow_unused=True)

    whole = second_order(lambda b, h, w: conv._SageFunction.apply(b, h, None, *w, False))
    want = second_order(lambda b, h, w: _plain(b, h, h[:b.num_dst_nodes()], *w))
    for a, b in zip(whole, want):
        if b is not None and float(b.norm()) > 0:
            assert a is not None and float((a - b).norm() / b.norm()) < 1e-12


def test_penalty_reaches_given_own_rows(operators):
    gen = torch.Generator().manual_seed(4)
    block = _block(30, 17, gen)
    w = [torch.randn(s, generator=gen, dtype=torch.float64).requires_grad_() for s in ((6, 5), (6, 5), (6,))]
    x = torch.randn((30, 5), generator=gen, dtype=torch.float64)
    own = torch.randn((17, 5), generator=gen, dtype=torch.float64).requires_grad_()
    got = []
    for out in (conv._SageFunction.apply(block, x, own, *w, False), _plain(block, x, own, *w)):
        g = torch.autograd.grad((out ** 3).sum(), w + [own], create_graph=True)
        got.append(torch.autograd.grad(sum((t ** 2).sum() for t in g), w + [own]))
    for a, b in zip(*got):
        assert float((a - b).norm() / b.norm()) < 1e-12
