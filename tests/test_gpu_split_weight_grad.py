"""The weight gradient in three bf16 parts a value (csrc/fgl_wgrad.hip) against float64: short and odd numbers of steps, tiles that the columns do not fill, many tiles
with several rounds of workgroups, strided rows with their column sums, and values that have no three parts."""
import pytest
import torch

from fastgl import _lib as L
from fastgl import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n", [(100, 64), (97, 200), (256, 47), (127, 129), (602, 256)])
def test_against_float64(cuda, m, n):
    gen = torch.Generator(device=cuda).manual_seed(m + n)
    for k in (1, 15, 16, 17, 63, 65, 127, 129, 1001, 8192, 30011):
        print("weight gradient", m, n, k, flush=True)
        a = torch.full((k, m + 3), float("nan"), device=cuda)[:, 1:m + 1]  # (what lies around the rows must not be read into the sums)
        a.copy_(torch.randn((k, m), generator=gen, device=cuda))
        b = torch.randn((k, n), generator=gen, device=cuda)
        got, sums = ops.weight_grad(a, b, column_sums=True)
        if m * n <= 65536 or k * k >= 256 * m * n:  # (else the library's)
            assert L.lib().fgl_product_last_kernel() == (b"wgrad_kernel in parts" if k >= 16 else b"wgrad_kernel")
        want, size = a.double().t() @ b.double(), a.double().abs().t() @ b.double().abs()
        # a step of 16 rows is right to 2^-24 of its largest sum or so, and k / 16 of them are added up in fp32: within (k / 16 + 16) 2^-24 of the magnitudes
        assert bool(((got.double() - want).abs() <= (k / 16 + 16) * 2.0 ** -24 * size).all())
        assert bool(((sums.double() - a.double().sum(0)).abs() <= (k / 16 + 16) * 2.0 ** -24 * a.double().abs().sum(0)).all())
        again = ops.weight_grad(a, b)
        assert torch.equal(got, again)


@pytest.mark.parametrize("m,n", [(100, 256), (256, 47), (64, 128)])
def test_few_rows_are_as_exact_as_fp32(cuda, m, n):
    gen = torch.Generator(device=cuda).manual_seed(m)
    a, b = torch.randn((15, m), generator=gen, device=cuda), torch.randn((15, n), generator=gen, device=cuda)
    assert torch.equal(ops.weight_grad(a[:1], b[:1]), a[0][:, None] * b[0])  # one product, rounded once
    for k in (2, 3, 15):
        want, size = a[:k].double().t() @ b[:k].double(), a[:k].double().abs().t() @ b[:k].double().abs()
        assert bool(((ops.weight_grad(a[:k], b[:k]).double() - want).abs() <= k * 2.0 ** -24 * size).all())  # (k products and k - 1 sums, each rounded once)


def test_errors_do_not_add_up_over_the_rows(cuda):
    """2-norm of the error over the result's: with the cut of the matrix instructions on one side it was 7e-7 here, that of fp32 sums is 3e-7."""
    gen = torch.Generator(device=cuda).manual_seed(3)
    a, b = torch.randn((107_000, 100), generator=gen, device=cuda), torch.randn((107_000, 256), generator=gen, device=cuda)
    want = a.double().t() @ b.double()
    ops.weight_grad(a, b)
    assert L.lib().fgl_product_last_kernel() == b"wgrad_kernel in parts"
    assert (ops.weight_grad(a, b).double() - want).norm() <= 2.8e-7 * want.norm()


def test_values_without_three_parts(cuda):
    k, m, n = 5000, 100, 128
    gen = torch.Generator(device=cuda).manual_seed(5)
    a, b = torch.randn((k, m), generator=gen, device=cuda), torch.randn((k, n), generator=gen, device=cuda) * 0.01
    a[70, 3], a[4000, 9], b[4999, 100] = float("inf"), float("nan"), float("-inf")
    a[:, 20] *= 1e-36      # (bits below bf16's last)
    a[17, 30] = 3.4e38     # (rounds to infinity in bf16)
    got, want = ops.weight_grad(a, b), a.double().t() @ b.double()
    assert L.lib().fgl_product_last_kernel() == b"wgrad_kernel in parts"
    odd = ~torch.isfinite(want)
    assert bool(odd[3].all()) and bool(odd[9].all()) and bool(odd[:, 100].all()) and int(odd.sum()) == 2 * n + m - 2
    assert torch.allclose(got[odd].double(), want[odd], rtol=0, atol=0, equal_nan=True)
    size = a.double().abs().t() @ b.double().abs()
    assert bool(((got.double() - want).abs() <= (k / 16 + 16) * 2.0 ** -24 * size + k * 2.0 ** -149)[~odd].all())


def _through_c(a, b, ws_bytes):
    """The C entry on a workspace of so many bytes: status, result."""
    lib, (k, m), n = L.lib(), a.shape, b.size(1)
    out, ws = torch.empty((m, n), dtype=a.dtype, device=a.device), torch.empty(ws_bytes, dtype=torch.uint8, device=a.device)
    dtype = L.F32 if a.dtype == torch.float32 else L.BF16
    rc = lib.fgl_weight_grad(a.data_ptr(), a.stride(0), b.data_ptr(), b.stride(0), k, m, n, dtype, out.data_ptr(), n, None, ws.data_ptr(), ws_bytes, L.stream_handle())
    return rc, out


@pytest.mark.parametrize("k,m,n,kernel", [(1000, 1000, 1000, b"wgrad_kernel"), (3000, 1000, 1000, b"wgrad_kernel in parts"), (1000, 602, 2000, b"wgrad_kernel"),
                                          (3000, 602, 2000, b"wgrad_kernel in parts"), (20_000, 100, 4000, b"wgrad_kernel"), (8000, 100, 4000, b"wgrad_kernel in parts"),
                                          (1000, 256, 256, b"wgrad_kernel in parts")])
def test_line_between_the_forms(cuda, k, m, n, kernel):
    """Few splits of k leave XCDs idle: many tiles and a short k are the fp32 form's."""
    gen = torch.Generator(device=cuda).manual_seed(k)
    a, b = torch.randn((k, m), generator=gen, device=cuda), torch.randn((k, n), generator=gen, device=cuda)
    rc, got = _through_c(a, b, L.lib().fgl_weight_grad_workspace_bytes(k, m, n))
    assert rc == 0 and L.lib().fgl_product_last_kernel() == kernel
    want, size = a.double().t() @ b.double(), a.double().abs().t() @ b.double().abs()
    assert bool(((got.double() - want).abs() <= (k / 16 + 16) * 2.0 ** -24 * size).all())


def test_workspace_of_the_fp32_form(cuda):
    """A caller whose workspace was sized for another k, of which the parts are not asked: the fp32 form, an error only below what that needs."""
    lib, k, m, n = L.lib(), 3000, 602, 1000
    gen = torch.Generator(device=cuda).manual_seed(9)
    a, b = torch.randn((k, m), generator=gen, device=cuda), torch.randn((k, n), generator=gen, device=cuda)
    whole, less = lib.fgl_weight_grad_workspace_bytes_for(k, m, n, L.F32), lib.fgl_weight_grad_workspace_bytes_for(k, m, n, L.BF16)
    assert less < whole
    want, size = a.double().t() @ b.double(), a.double().abs().t() @ b.double().abs()
    for ws_bytes, kernel in ((whole, b"wgrad_kernel in parts"), (less, b"wgrad_kernel")):
        rc, got = _through_c(a, b, ws_bytes)
        assert rc == 0 and lib.fgl_product_last_kernel() == kernel
        assert bool(((got.double() - want).abs() <= (k / 16 + 16) * 2.0 ** -24 * size).all())
    assert _through_c(a, b, 1024)[0] != 0


@pytest.mark.parametrize("k", [64, 5000, 30011])
def test_values_whose_last_bits_bf16_has_not(cuda, k):
    """Tiny values beside large ones in one column: they are lost in three parts (below 2^-133) and count where the others meet zeros."""
    m, n = 100, 256
    gen = torch.Generator(device=cuda).manual_seed(k)
    a, b = torch.randn((k, m), generator=gen, device=cuda), torch.randn((k, n), generator=gen, device=cuda)
    b[torch.rand((k, n), generator=gen, device=cuda) < 0.001] *= 1e-37  # (which do not count)
    few = 2.0 ** -120 * (1 + 2.0 ** -20)
    a[:, 20] = 0
    a[0, 20], a[k - 1, 20] = 1, few
    b[0, 7], b[k - 1, 7] = 0, 2.0 ** 110
    b[:, 200] = 0
    b[3, 200], b[k // 2, 200] = 1, few
    a[3, 50], a[k // 2, 50] = 0, 2.0 ** 110
    got = ops.weight_grad(a, b)
    assert L.lib().fgl_product_last_kernel() == b"wgrad_kernel in parts"
    assert float(got[20, 7]) == float(got[50, 200]) == few * 2.0 ** 110
    want, size = a.double().t() @ b.double(), a.double().abs().t() @ b.double().abs()
    keep = torch.ones((m, n), dtype=torch.bool, device=cuda)
    keep[50], keep[:, 7] = False, False
    assert bool(((got.double() - want).abs() <= (k / 16 + 16) * 2.0 ** -24 * size)[keep].all())
