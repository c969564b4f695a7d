"""Products of more than 8e9 multiplications on both sides of ops._long_product_is_the_kernels, against float64."""
import pytest
import torch

from fastgl import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("dtype,m,k,n,kernels", [  # (kernels: in the plain and in the transposed layout)
    (torch.float32, 1_300_001, 100, 66, (False, False)), (torch.float32, 1_300_001, 100, 64, (False, False)), (torch.float32, 5_000_001, 32, 64, (True, True)),
    (torch.float32, 2_500_000, 101, 33, (False, True)), (torch.float32, 1_300_001, 64, 100, (True, True)), (torch.float32, 1_100_001, 90, 90, (True, False)),
    (torch.float32, 700_001, 96, 130, (False, False)), (torch.float32, 300_001, 101, 300, (True, False)), (torch.float32, 300_001, 129, 250, (False, False)),
    (torch.bfloat16, 1_300_001, 100, 64, (True, True)), (torch.bfloat16, 1_000_003, 128, 64, (True, False)), (torch.bfloat16, 1_000_003, 96, 96, (False, False)),
    (torch.bfloat16, 500_001, 100, 201, (True, False))])
def test_long_products(cuda, dtype, m, k, n, transposed, kernels):
    print("long product", dtype, m, k, n, transposed, flush=True)
    gen = torch.Generator(device=cuda).manual_seed(m)
    a = torch.randn((m, k), generator=gen, device=cuda).to(dtype)
    b = torch.randn((n, k) if transposed else (k, n), generator=gen, device=cuda).to(dtype)
    assert m * k * n > 8 * 10 ** 9
    assert (ops._forms_row_product(a, b, transposed, m, k, n) is not None) == kernels[transposed]
    got = ops.row_product(a, b, transposed)
    for rows in (slice(0, 300), slice(m // 2, m // 2 + 300), slice(m - 300, m)):
        x, w = a[rows].double(), (b.t() if transposed else b).double()
        bound = (k + 2) * 2.0 ** -24 * (x.abs() @ w.abs())
        want = x @ w
        if dtype == torch.bfloat16:
            bound = bound + want.abs() * 2.0 ** -8
        assert bool(((got[rows].double() - want).abs() <= bound).all())
