"""fgl_weight_grad (the k-splitting product behind d_w of every layer) against a float64 product, at the edges of its tiles and
steps: columns that pad a tile of 32, 64 or 128, single rows, short last steps, odd row strides, one and many k splits."""
import pytest
import torch

import fastgl
from fastgl import _lib as L
from fastgl import ops

pytestmark = pytest.mark.gpu


def _product(a, b, want_sums=True):
    lib = fastgl.lib()
    (k, m), n = a.shape, b.shape[1]
    c = torch.full((m, n), 7.0, dtype=a.dtype, device=a.device)
    sums = torch.full((m,), 7.0, dtype=a.dtype, device=a.device)
    ws = torch.empty(lib.fgl_weight_grad_workspace_bytes(k, m, n), dtype=torch.uint8, device=a.device)
    L.check(lib.fgl_weight_grad(a.data_ptr(), a.stride(0), b.data_ptr(), b.stride(0), k, m, n,
                                L.F32 if a.dtype == torch.float32 else L.BF16, c.data_ptr(), n, sums.data_ptr() if want_sums else None,
                                ws.data_ptr(), ws.numel(), L.stream_handle()))
    return c, sums


def _check(got, a, b, k):
    # The sums are fp32 on both dtypes (products of bf16 values are exact in fp32): with ~N(0,1) operands the partial sums are
    # ~sqrt(k) and the chains of additions a few hundred long, 6e-6 sqrt(k) in all.  A bf16 result is then rounded once: at most
    # half a unit in the last of its eight places, 2^-8 of the value.
    want = a.double().t() @ b.double()
    limit = 6e-6 * max(1.0, k ** 0.5) + (want.abs() * 2.0 ** -8 if a.dtype == torch.bfloat16 else 0.0)
    assert ((got.double() - want).abs() <= limit).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("m,n", [(1, 1), (3, 2), (16, 47), (33, 64), (64, 33), (100, 256), (127, 130), (128, 128), (602, 17), (65, 7),
                                 (256, 256), (34, 300)])
def test_matches_float64(cuda, dtype, m, n):
    gen = torch.Generator(device=cuda).manual_seed(m * 1000 + n)
    for k in (1, 7, 8, 9, 31, 32, 63, 64, 65, 255, 256, 1000, 4097, 20011):
        a = torch.randn((k, m), generator=gen, device=cuda).to(dtype)
        b = torch.randn((k, n), generator=gen, device=cuda).to(dtype)
        c, sums = _product(a, b)
        _check(c, a, b, k)
        _check(sums[:, None], a, torch.ones((k, 1), dtype=dtype, device=cuda), k)
        again, _ = _product(a, b, want_sums=False)
        assert torch.equal(c, again)  # the same bits on every run, with or without the column sums


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_row_strides_and_rows_around_are_left_alone(cuda, dtype):
    gen = torch.Generator(device=cuda).manual_seed(3)
    # slices of wider arrays whose other columns are not numbers: nothing of them may reach the result
    wide_a = torch.full((501, 75), float("nan"), dtype=dtype, device=cuda)
    wide_b = torch.full((501, 140), float("nan"), dtype=dtype, device=cuda)
    for ca, cb, m, n in ((0, 0, 33, 64), (1, 3, 50, 101), (42, 100, 33, 40)):
        a, b = wide_a[:500, ca:ca + m], wide_b[:500, cb:cb + n]
        a.copy_(torch.randn((500, m), generator=gen, device=cuda))
        b.copy_(torch.randn((500, n), generator=gen, device=cuda))
        c, sums = _product(a, b)
        _check(c, a, b, 500)
        _check(sums[:, None], a, torch.ones((500, 1), dtype=dtype, device=cuda), 500)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_linear_layer_gradients(cuda, dtype):
    # the layer behind SAGE and GAT against nn.Linear on the same numbers, gradients of all three operands
    from fastgl.conv import _Linear
    torch.manual_seed(0)
    ours = _Linear(70, 90).to(cuda, dtype)
    theirs = torch.nn.Linear(70, 90).to(cuda, dtype)
    theirs.load_state_dict(ours.state_dict())
    x = torch.randn(3000, 70, device=cuda).to(dtype)
    g = torch.randn(3000, 90, device=cuda).to(dtype)
    got, want = [], []
    for layer, out in ((ours, got), (theirs, want)):
        xi = x.clone().requires_grad_()
        y = layer(xi)
        y.backward(g)
        out += [y.detach(), xi.grad, layer.weight.grad, layer.bias.grad]
    for a, b in zip(got, want):  # both sides round once to the dtype; fp32 sums of 3000 terms in another order
        assert (a.double() - b.double()).norm() / b.double().norm() <= (3e-6 if dtype == torch.float32 else 6e-3)
    # a second derivative still runs (the gradient's own graph)
    xi = x.float().clone().requires_grad_()
    layer = _Linear(70, 90).to(cuda)
    (dx,) = torch.autograd.grad(layer(xi).square().sum(), xi, create_graph=True)
    dx.square().sum().backward()
    assert xi.grad is not None and torch.isfinite(xi.grad).all()


def test_rule_of_the_dispatch():
    assert ops._splits_k(300, 64, 47) and ops._splits_k(105_000, 100, 256) and ops._splits_k(8192, 602, 256)
    assert not ops._splits_k(8192, 1024, 1024) and not ops._splits_k(2000, 256, 1024)
