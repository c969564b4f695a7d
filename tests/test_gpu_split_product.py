"""fp32 products over rows on the bf16 matrix cores (csrc/fgl_split_product.hip) against float64, at the edges of their tiles: row tiles of 32, 32, 64 and 128
columns a workgroup, steps of 16 k that are odd or even in number and end with k, k too long for one width of B in LDS; and values that have no three bf16 parts."""
import pytest
import torch

from fastgl import _lib as L
from fastgl import ops

pytestmark = pytest.mark.gpu

# (rows, k, columns) on both sides of the line between the kernels: those that are in parts, and those that the fp32 instructions form
IN_PARTS = [(480_001, 33, 63), (180_001, 48, 130), (440_001, 49, 31), (100_001, 64, 129), (26_001, 100, 256), (95_003, 96, 66), (6_417, 256, 300), (6_500, 416, 250),
            (6_500, 417, 250), (50_001, 832, 33), (2000, 256, 1100), (33_269, 100, 128), (1_000_001, 17, 65), (400_003, 32, 40), (5_000_001, 12, 90),
            (476_628, 100, 6), (24_000, 256, 72), (200_001, 56, 127), (147_000, 27, 256), (700_001, 18, 100)]
PLAIN = [(1_600_001, 1, 128), (450_017, 7, 65), (210_031, 15, 64), (210_001, 16, 64), (400_033, 17, 31), (97_001, 33, 63), (909_001, 8, 33), (50_001, 833, 33),
         (1990, 256, 1200), (4000, 400, 400), (32_003, 96, 66), (5_000_001, 3, 90), (1_000_001, 16, 97), (1_000_001, 24, 32), (5_500, 256, 256), (1_000_001, 32, 102),
         (200_001, 55, 127), (180_001, 48, 129), (300_001, 32, 380)]


def _kernel():
    return L.lib().fgl_product_last_kernel()


def _check(got, want, bound):
    assert bool(((got.double() - want).abs() <= bound).all())


@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("m,k,n", IN_PARTS + PLAIN)
def test_split_product(cuda, m, k, n, transposed):
    print("split product", m, k, n, transposed, flush=True)
    gen = torch.Generator(device=cuda).manual_seed(m + k + n)
    a = torch.full((m, k + 3), float("nan"), device=cuda)[:, 1:k + 1]  # (rows that start on no vector's boundary; what lies around must not be read into the sums)
    a.copy_(torch.randn((m, k), generator=gen, device=cuda))
    b = torch.randn((n, k) if transposed else (k, n), generator=gen, device=cuda)
    bias = torch.randn(n, generator=gen, device=cuda)
    w = (b.t() if transposed else b).double()
    got, plus, through_c = ops.row_product(a, b, transposed), ops.row_product(a, b, transposed, bias), torch.empty((m, n), device=cuda)
    L.check(L.lib().fgl_row_product(a.data_ptr(), k + 3, b.data_ptr(), b.size(1), int(transposed), m, k, n, L.F32, None, through_c.data_ptr(), n, L.stream_handle()))
    assert _kernel() == (b"split_product_kernel" if (m, k, n) in IN_PARTS else b"row_product_kernel")
    for rows in (slice(0, 5000), slice(m // 2, m // 2 + 5000), slice(max(m - 5000, 0), m)):
        x = a[rows].double()
        # three parts of eight bits each: the products that are left out are below 2^-26, what a matrix instruction cuts off below 2^-25 of a chunk's sum, and k / 32
        # sums are rounded: within the (k + 2) 2^-24 of the magnitudes that k fp32 products and sums are given
        want, bound = x @ w, (k + 2) * 2.0 ** -24 * (x.abs() @ w.abs() + bias.double().abs())
        _check(got[rows], want, bound)
        _check(through_c[rows], want, bound)
        _check(plus[rows], want + bias.double(), bound)


def test_one_term_is_rounded_once(cuda):
    gen = torch.Generator(device=cuda).manual_seed(2)
    a, b = torch.randn((1_700_001, 1), generator=gen, device=cuda), torch.randn((1, 128), generator=gen, device=cuda)
    assert torch.equal(ops.row_product(a, b), a * b)


@pytest.mark.parametrize("m,k0,k1,n", [(120_001, 100, 33, 65), (13_501, 256, 128, 128), (30_001, 16, 400, 64), (160_001, 7, 100, 65), (150_001, 100, 1, 65),
                                       (250_003, 15, 40, 64)])
def test_sums_and_additions(cuda, m, k0, k1, n):
    gen = torch.Generator(device=cuda).manual_seed(m)
    a0, a1 = (torch.randn((m, k), generator=gen, device=cuda) for k in (k0, k1))
    b0, b1 = (torch.randn((n, k), generator=gen, device=cuda) for k in (k0, k1))
    bias, base = torch.randn(n, generator=gen, device=cuda), torch.randn((m + 5, n), generator=gen, device=cuda)
    want, size = a0.double() @ b0.double().t() + a1.double() @ b1.double().t() + bias.double(), a0.double().abs() @ b0.double().abs().t() + a1.double().abs() @ b1.double().abs().t()
    got = ops.row_product_sum(a0, b0, a1, b1, bias)
    assert _kernel() == b"split_product_kernel"
    _check(got, want, (k0 + k1 + 2) * 2.0 ** -24 * (size + bias.double().abs()))
    w = b0.t().contiguous()
    got = ops.row_product_add_(base.clone(), a0, w)
    assert (_kernel() == b"split_product_kernel") == (k0 >= 100)
    assert torch.equal(got[m:], base[m:])
    size = a0.double().abs() @ w.double().abs() + base[:m].double().abs()
    _check(got[:m], a0.double() @ w.double() + base[:m].double(), (k0 + 2) * 2.0 ** -24 * size)


@pytest.mark.parametrize("transposed", [False, True])
def test_values_without_three_parts(cuda, transposed):
    m, k, n = 90_000, 100, 64
    gen = torch.Generator(device=cuda).manual_seed(5)
    a, b = torch.randn((m, k), generator=gen, device=cuda), torch.randn((n, k) if transposed else (k, n), generator=gen, device=cuda)
    clean = ops.row_product(a, b, transposed)
    assert _kernel() == b"split_product_kernel"
    a[70, 3], a[1000, 99], a[1000, 5], a[5000, 0], a[5001, 98] = float("inf"), float("inf"), float("-inf"), float("nan"), float("-inf")
    a[9000] = 3.4e38 * torch.rand(k, generator=gen, device=cuda) ** 0.01  # (rounds to infinity in bf16)
    b.mul_(0.01)
    a[20000] *= 1e-36  # (bits below bf16's last)
    a[30000] *= 1e-42
    got, w = ops.row_product(a, b, transposed), (b.t() if transposed else b).double()
    want = a.double() @ w
    for r in (70, 1000, 5000, 5001):  # (row 1000: inf * w - inf * w', infinite or not a number by the weights' signs)
        assert not bool(torch.isfinite(got[r]).any()) and torch.allclose(got[r].double(), want[r], rtol=0, atol=0, equal_nan=True)
    rest = torch.tensor([r for r in range(m) if r not in (70, 1000, 5000, 5001)], device=cuda)
    # (subnormal operands and results: each rounded to a multiple of 2^-149 at most once a term)
    _check(got[rest], want[rest], (k + 2) * 2.0 ** -24 * (a[rest].double().abs() @ w.abs()) + (k + 2) * 2.0 ** -149)
    neighbours = torch.cat((torch.arange(0, 70), torch.arange(1024, 4992), torch.arange(31000, m))).to(cuda)
    _check(got[neighbours], clean[neighbours].double() * 0.01, (k + 4) * 2.0 ** -23 * (a[neighbours].double().abs() @ w.abs()))


@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("m,k,n", [(90_000, 100, 64), (100_001, 64, 129), (6_500, 416, 250), (6_500, 417, 250)])
def test_values_whose_last_bits_bf16_has_not(cuda, m, k, n, transposed):
    """Tiny values beside large ones in one row or column: they are lost in three parts (below 2^-133) and count where the others meet zeros."""
    gen = torch.Generator(device=cuda).manual_seed(6)
    a, b = torch.randn((m, k), generator=gen, device=cuda), torch.randn((k, n), generator=gen, device=cuda)
    tiny = torch.rand((m, k), generator=gen, device=cuda) < 0.01
    a[tiny] *= 1e-37                      # (which do not count)
    few = 2.0 ** -120 * (1 + 2.0 ** -20)  # 21 bits, of which bf16 holds 14
    rows = [5, 1000, m - 1]
    a[rows] = 0
    a[rows, 0], a[rows, 1] = 1, few
    b[0, 7], b[1, 7] = 0, 2.0 ** 110
    b[:, n - 1] = 0                       # the same in a column
    b[2, n - 1], b[k - 1, n - 1] = 1, few
    a[77], a[77, k - 1] = 0, 2.0 ** 110
    w = b.t().contiguous() if transposed else b
    got = ops.row_product(a, w, transposed)
    assert _kernel() == b"split_product_kernel"
    want = a.double() @ b.double()
    one = torch.cat((got[rows, 7], got[77, n - 1:]))
    assert bool((one == few * 2.0 ** 110).all())
    rest = torch.ones((m, n), dtype=torch.bool, device=cuda)
    rest[77], rest[:, 7] = False, False
    assert bool(((got.double() - want).abs() <= (k + 2) * 2.0 ** -24 * (a.double().abs() @ b.double().abs()))[rest].all())
    # results that are subnormal: each term and each sum is rounded to a multiple of 2^-149 once
    a, b = torch.randn((m, k), generator=gen, device=cuda) * 1e-28, torch.randn((k, n), generator=gen, device=cuda) * 1e-12
    got = ops.row_product(a, b.t().contiguous() if transposed else b, transposed)
    assert bool(((got.double() - a.double() @ b.double()).abs() <= (k + 2) * 2.0 ** -149).all())


@pytest.mark.parametrize("m,k,n,split", [(1_300_001, 100, 64, True), (1_300_001, 100, 66, False), (8192, 256, 602, True), (3000, 256, 602, False), (8192, 602, 256, False),
                                         (2048, 256, 2000, True), (1999, 256, 2000, False), (3000, 256, 1000, False), (3000, 100, 2000, True), (200, 256, 20000, False),
                                         (300_001, 200, 160, False), (600_001, 384, 40, False)])
def test_products_beyond_the_general_line(cuda, m, k, n, split):
    print("long or wide product", m, k, n, flush=True)
    gen = torch.Generator(device=cuda).manual_seed(m)
    a = torch.randn((m, k), generator=gen, device=cuda)
    for transposed in (False, True):
        b = torch.randn((n, k) if transposed else (k, n), generator=gen, device=cuda)
        assert ops._forms_row_product(a, b, transposed, m, k, n) is None
        assert (ops._forms_split_product(a, b, transposed, m, k, n) is not None) == split
        got, w = ops.row_product(a, b, transposed), (b.t() if transposed else b).double()
        assert not split or _kernel() == b"split_product_kernel"
        for rows in (slice(0, 1000), slice(max(m - 1000, 0), m)):
            x = a[rows].double()
            _check(got[rows], x @ w, (k + 2) * 2.0 ** -24 * (x.abs() @ w.abs()))


@pytest.mark.parametrize("m,k,n", [(2000, 256, 16384), (2000, 256, 16385), (2037, 256, 20000), (2000, 100, 32768), (2000, 100, 32769), (2048, 100, 40000),
                                   (2000, 832, 8192), (2000, 832, 8193), (2000, 500, 20000), (2000, 100, 65536)])
def test_more_tiles_along_n_than_the_chip_holds(cuda, m, k, n):
    """Products with so many columns that the workgroups of one row tile each are more than the chip takes at a time."""
    print("wide product", m, k, n, flush=True)
    gen = torch.Generator(device=cuda).manual_seed(n)
    a = torch.randn((m, k), generator=gen, device=cuda)
    lib = L.lib()
    for transposed in (False, True):
        b = torch.randn((n, k) if transposed else (k, n), generator=gen, device=cuda)
        w = (b.t() if transposed else b).double()
        want, bound = a.double() @ w, (k + 2) * 2.0 ** -24 * (a.double().abs() @ w.abs())
        _check(ops.row_product(a, b, transposed), want, bound)
        got = torch.full((m, n), float("nan"), device=cuda)  # (the C entry itself: from Python some of these are the library's)
        L.check(lib.fgl_row_product(a.data_ptr(), k, b.data_ptr(), k if transposed else n, int(transposed), m, k, n, L.F32, None, got.data_ptr(), n,
                                    L.stream_handle()))
        assert _kernel() == b"split_product_kernel"
        _check(got, want, bound)


def _time(f):
    """The shortest of a few runs of ten calls, in milliseconds a call."""
    best = float("inf")
    f()
    for _ in range(5):
        begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        begin.record()
        for _ in range(10):
            f()
        end.record()
        end.synchronize()
        best = min(best, begin.elapsed_time(end) / 10)
    return best


@pytest.mark.parametrize("m,k,fewer,more", [(100_396, 128, 376, 512), (100_396, 64, 896, 1024), (80_001, 256, 1064, 1280)])
def test_fewer_columns_take_no_longer(cuda, m, k, fewer, more):
    """Workgroups of one more row block than the chip holds take as long as a second round: 6 and 17 tiles of columns took 1.4 and 1.3 times what 8 and 20 do."""
    gen = torch.Generator(device=cuda).manual_seed(k)
    a, b = torch.randn((m, k), generator=gen, device=cuda), torch.randn((more, k), generator=gen, device=cuda)
    w = b[:fewer].contiguous()
    got = ops.row_product(a, w, True)
    assert _kernel() == b"split_product_kernel"
    for rows in (slice(0, 1000), slice(m - 1000, m)):
        x = a[rows].double()
        _check(got[rows], x @ w.double().t(), (k + 2) * 2.0 ** -24 * (x.abs() @ w.double().abs().t()))
    assert _time(lambda: ops.row_product(a, w, True)) < 1.05 * _time(lambda: ops.row_product(a, b, True))


@pytest.mark.parametrize("first,ldc", [(0, 132), (1, 132), (2, 132), (0, 130), (3, 131), (0, 127)])
@pytest.mark.parametrize("m,k,n", [(180_001, 60, 127), (100_001, 100, 126), (50_001, 832, 33)])
def test_rows_of_every_alignment(cuda, m, k, n, first, ldc):
    """Results of which every row starts on a vector of four, of two or of one value: all of them, and nothing beside them."""
    gen = torch.Generator(device=cuda).manual_seed(ldc)
    a, b, bias = (torch.randn(s, generator=gen, device=cuda) for s in ((m, k), (k, n), (n,)))
    base = torch.randn(m * ldc + 8, generator=gen, device=cuda)
    want = base.clone().as_strided((m, n), (ldc, 1), first)
    w, lib = b.double(), L.lib()
    for transposed in (False, True):
        x = b.t().contiguous() if transposed else b
        for add in (False, True):
            buf = base.clone()
            out = buf.as_strided((m, n), (ldc, 1), first)
            if add:
                L.check(lib.fgl_row_product_add(a.data_ptr(), k, x.data_ptr(), x.size(1), int(transposed), m, k, n, L.F32, out.data_ptr(), ldc, L.stream_handle()))
            else:
                L.check(lib.fgl_row_product(a.data_ptr(), k, x.data_ptr(), x.size(1), int(transposed), m, k, n, L.F32, bias.data_ptr(), out.data_ptr(), ldc,
                                            L.stream_handle()))
            assert _kernel() == b"split_product_kernel"
            for rows in (slice(0, 3000), slice(m - 3000, m)):
                more = want[rows].double() if add else bias.double()
                r = a[rows].double()
                _check(out[rows], r @ w + more, (k + 2) * 2.0 ** -24 * (r.abs() @ w.abs() + more.abs()))
            out.copy_(base.as_strided((m, n), (ldc, 1), first))
            assert torch.equal(buf, base)


@pytest.mark.parametrize("n", [125, 126])
def test_columns_that_fill_no_vectors(cuda, n):
    """Misaligned stores of four values a lane took 1.7 times as long as aligned ones."""
    gen = torch.Generator(device=cuda).manual_seed(n)
    a, b = torch.randn((600_000, 64), generator=gen, device=cuda), torch.randn((128, 64), generator=gen, device=cuda)
    w = b[:n].contiguous()
    assert n == 125 or _time(lambda: ops.row_product(a, w, True)) < 1.45 * _time(lambda: ops.row_product(a, b, True))
    assert _time(lambda: ops.row_product(a, w, True)) < 1.6 * _time(lambda: ops.row_product(a, b, True))


def test_an_addition_costs_what_it_reads(cuda):
    """C read a row at a time, each behind the stores of the row before, made this 3.0 times the product alone; its bytes are 1.4 times as many."""
    gen = torch.Generator(device=cuda).manual_seed(47)
    a, b, out = (torch.randn(s, generator=gen, device=cuda) for s in ((895_000, 64), (64, 47), (895_000, 47)))
    assert _time(lambda: ops.row_product_add_(out, a, b)) < 2.0 * _time(lambda: ops.row_product(a, b))
    assert _kernel() == b"split_product_kernel"


@pytest.mark.parametrize("e", [12, 13, 14, 20])
def test_parts_below_the_smallest_normal_number(cuda, e):
    """A value whose second part is subnormal in bf16 (up to e = 13 none of its bits are lost there) and the only one that counts: its product is exact."""
    m, k, n = 100_001, 100, 64
    few = 2.0 ** -120 * (1 + 2.0 ** -e)
    a, b = torch.zeros((m, k), device=cuda), torch.zeros((k, n), device=cuda)
    a[:, 7], b[7] = few, 2.0 ** 110
    got = ops.row_product(a, b)
    assert _kernel() == b"split_product_kernel" and bool((got == few * 2.0 ** 110).all())
    a[:, 7], b[7] = 2.0 ** 110, few
    assert bool((ops.row_product(a, b) == few * 2.0 ** 110).all())
    x, y = torch.zeros((5000, 100), device=cuda), torch.zeros((5000, 256), device=cuda)
    for row in (0, 4999):
        x.zero_(), y.zero_()
        x[row], y[row] = few, 2.0 ** 110
        assert bool((ops.weight_grad(x, y) == few * 2.0 ** 110).all()) and _kernel() == b"wgrad_kernel in parts"
