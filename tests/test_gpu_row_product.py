"""ops.row_product against the product in float64, at the edges of its tiles: columns in vectors of 1, 2 and 4 times 32 lanes, row tiles of
32 and 64, steps of 8 (fp32) and 16 (bf16) k with a remainder, both layouts of the weight."""
import pytest
import torch

import fastgl
from fastgl import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

SHAPES = [(1, 1, 1), (31, 7, 3), (32, 8, 32), (33, 9, 33), (64, 16, 64), (129, 100, 64), (1000, 602, 47), (40000, 17, 128), (70001, 100, 256),
          (150000, 33, 64), (9000, 16, 300)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("m,k,n", SHAPES)
def test_row_product(m, k, n, transposed, dtype):
    gen = torch.Generator(device=DEV).manual_seed(m + k + n)
    pad = k + k % 2  # (bf16 rows on word boundaries; what lies behind k must not be read into the sums)
    def rows(r, c, width):
        x = torch.randn((r, width), generator=gen, device=DEV)
        x[:, c:] = float("nan")
        return x.to(dtype)[:, :c]
    a = rows(m, k, pad)
    b = rows(n, k, pad) if transposed else rows(k, n, n)
    bias = torch.randn(n, generator=gen, device=DEV).to(dtype)
    assert ops._forms_row_product(a, b, transposed, m, k, n)
    ad, bd = a.double(), (b.t() if transposed else b).double()
    # k fp32 products and sums: each result is off by at most (k + 1) eps of the sum of the products' magnitudes; bf16 rounds the result once
    bound = (k + 2) * 2.0 ** -24 * (ad.abs() @ bd.abs() + bias.double().abs())
    for use_bias in (False, True):
        want = ad @ bd + (bias.double() if use_bias else 0)
        got = ops.row_product(a, b, transposed, bias if use_bias else None)
        assert got.shape == (m, n) and got.dtype == dtype
        limit = bound + (want.abs() * 2.0 ** -8 if dtype == torch.bfloat16 else 0)
        assert bool(((got.double() - want).abs() <= limit).all())


def test_row_product_forms_left_to_torch():
    a = torch.randn(40, 7, device=DEV).bfloat16()  # rows on odd element boundaries
    w = torch.randn(7, 16, device=DEV).bfloat16()
    assert not ops._forms_row_product(a, w, False, 40, 7, 16)
    assert torch.equal(ops.row_product(a, w), torch.mm(a, w))
    x, p = torch.randn(40, 8, device=DEV), torch.randn(8, 16, device=DEV, requires_grad=True)
    assert ops.row_product(x, p).requires_grad  # a graph is being recorded
    assert ops.row_product(x.new_empty((0, 8)), p.detach()).shape == (0, 16)
    with pytest.raises(RuntimeError):
        ops.row_product(x, p[:4])
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert ops.row_product(x, p.detach()).dtype == torch.bfloat16


def test_linear_without_gradients():
    lin = fastgl.conv._Linear(100, 47).to(DEV)
    x = torch.randn(333, 100, device=DEV)
    with torch.no_grad():
        want = torch.nn.functional.linear(x.double(), lin.weight.double(), lin.bias.double())
        assert torch.allclose(lin(x).double(), want, rtol=1e-5, atol=1e-5)
        assert torch.func.vmap(lin)(x[None]).shape == (1, 333, 47)  # watched tensors keep torch's operator
        with torch.autograd.forward_ad.dual_level():
            out = lin(torch.autograd.forward_ad.make_dual(x, torch.ones_like(x)))
            assert torch.autograd.forward_ad.unpack_dual(out).tangent is not None


def test_linear_with_gradients_under_transforms():
    """What torch's operator can do with a gradient being recorded, the layer still can: vmap, torch.func, forward mode, tracing."""
    lin = fastgl.conv._Linear(20, 7).to(DEV)
    x = torch.randn(33, 20, device=DEV)
    with torch.enable_grad():
        want = torch.nn.functional.linear(x, lin.weight, lin.bias)
        assert torch.func.vmap(lin)(x[None]).shape == (1, 33, 7)
        g = torch.func.grad(lambda p: torch.func.functional_call(lin, p, (x,)).sum())(dict(lin.named_parameters()))
        assert torch.allclose(g["weight"], x.sum(0).expand(7, 20), rtol=1e-4, atol=1e-4)
        with torch.autograd.forward_ad.dual_level():
            out = lin(torch.autograd.forward_ad.make_dual(x, torch.ones_like(x)))
            assert torch.autograd.forward_ad.unpack_dual(out).tangent is not None
        traced = torch.jit.trace(lin, (x,))
        assert torch.allclose(traced(x[:5]), want[:5], rtol=1e-4, atol=1e-4)
