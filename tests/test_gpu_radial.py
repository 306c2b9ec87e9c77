"""`radial_linear`: the matrix-core kernel of the radial network's last layer against the same
product in float64 (tolerance: float32 sums of `inner` terms)."""

import pytest
import torch

from e3j_amd import _lib
from e3j_amd.radial import radial_linear

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("inner", [8, 16, 32, 64, 128])
@pytest.mark.parametrize("edges,n", [(1, 32), (31, 64), (256, 1472), (257, 2944), (1000, 96)])
def test_forward_matches_the_float64_product(inner, edges, n):
    g = torch.Generator(device="cuda").manual_seed(inner * 1000 + edges)
    h = torch.randn(edges, inner, device="cuda", generator=g)
    w = torch.randn(inner, n, device="cuda", generator=g)
    s = radial_linear(h, w)
    want = h.double() @ w.double()
    bound = 1e-6 + 1e-5 * want.abs() + 8 * 2.0 ** -24 * (h.double().abs() @ w.double().abs())
    assert s.shape == (edges, n) and s.dtype == torch.float32
    assert bool(((s.double() - want).abs() <= bound).all())


@pytest.mark.parametrize("inner", [32, 64, 128])
def test_every_row_and_column_lands_in_its_place(inner):
    """h = one-hot rows, w = distinct integers: s[e, :] must be row (e mod inner) of w exactly
    (also on the kernels that split their operands three ways: integers below 2^24 split exactly)."""
    edges, n = 333, 160
    h = torch.zeros(edges, inner, device="cuda")
    h[torch.arange(edges), torch.arange(edges) % inner] = 1.0
    w = torch.arange(inner * n, device="cuda", dtype=torch.float32).reshape(inner, n)
    assert torch.equal(radial_linear(h, w), w[torch.arange(edges, device="cuda") % inner])


def test_gradients_and_errors():
    g = torch.Generator(device="cuda").manual_seed(5)
    h = torch.randn(100, 32, device="cuda", generator=g, requires_grad=True)
    w = torch.randn(32, 64, device="cuda", generator=g, requires_grad=True)
    ds = torch.randn(100, 64, device="cuda", generator=g)
    dh, dw = torch.autograd.grad(radial_linear(h, w), (h, w), ds)
    torch.testing.assert_close(dh, ds @ w.detach().t(), rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(dw, h.detach().t() @ ds, rtol=1e-5, atol=1e-5)
    assert radial_linear(h[:0], w).shape == (0, 64)
    with pytest.raises(ValueError, match="multiple of 32"):
        radial_linear(h, w[:, :40])
    with pytest.raises(ValueError):
        radial_linear(h[:, :24], w[:24])
    lib = _lib.load()
    assert lib.e3j_amd_radial_linear_fwd(None, None, None, 4, 24, 64, None) == _lib.UNIMPLEMENTED
    assert lib.e3j_amd_radial_linear_fwd(None, None, None, 4, 32, 64, None) == _lib.INVALID_ARGUMENT


@pytest.mark.parametrize("inner", [8, 16, 32, 64, 128])
@pytest.mark.parametrize("edges,n", [(1, 32), (70, 128), (4099, 1472), (20001, 96)])
def test_weight_gradient_matches_the_float64_product_and_repeats(inner, edges, n):
    g = torch.Generator(device="cuda").manual_seed(inner * 31 + edges)
    h = torch.randn(edges, inner, device="cuda", generator=g)
    w = torch.randn(inner, n, device="cuda", generator=g, requires_grad=True)
    ds = torch.randn(edges, n, device="cuda", generator=g)
    (dw,) = torch.autograd.grad(radial_linear(h, w), (w,), ds)
    want = h.double().t() @ ds.double()
    bound = 1e-6 + 1e-5 * want.abs() + 16 * 2.0 ** -24 * (h.double().abs().t() @ ds.double().abs())
    assert dw.shape == (inner, n)
    assert bool(((dw.double() - want).abs() <= bound).all())
    (again,) = torch.autograd.grad(radial_linear(h, w), (w,), ds)
    assert torch.equal(dw, again)   # fixed summation order over the edges


def test_second_derivative_goes_through_the_library_products():
    g = torch.Generator(device="cuda").manual_seed(9)
    h = torch.randn(50, 16, device="cuda", generator=g, requires_grad=True)
    w = torch.randn(16, 64, device="cuda", generator=g, requires_grad=True)
    ds = torch.randn(50, 64, device="cuda", generator=g, requires_grad=True)
    dh, dw = torch.autograd.grad(radial_linear(h, w), (h, w), ds, create_graph=True)
    (dds,) = torch.autograd.grad((dh.sum() + dw.sum()), (ds,))
    want = (torch.ones_like(dh) @ w + h @ torch.ones_like(dw)).detach()
    torch.testing.assert_close(dds, want, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("inner", [32, 64, 128])
@pytest.mark.parametrize("edges,n", [(1, 32), (33, 64), (257, 1472), (1000, 2944)])
def test_input_gradient_matches_the_float64_product(inner, edges, n):
    g = torch.Generator(device="cuda").manual_seed(inner * 77 + edges)
    h = torch.randn(edges, inner, device="cuda", generator=g, requires_grad=True)
    w = torch.randn(inner, n, device="cuda", generator=g)
    ds = torch.randn(edges, n, device="cuda", generator=g)
    (dh,) = torch.autograd.grad(radial_linear(h, w), (h,), ds)
    want = ds.double() @ w.double().t()
    bound = 1e-6 + 1e-5 * want.abs() + 16 * 2.0 ** -24 * (ds.double().abs() @ w.double().abs().t())
    assert dh.shape == (edges, inner)
    assert bool(((dh.double() - want).abs() <= bound).all())
    # one-hot cotangent rows pick rows of w^T exactly (integers split exactly)
    wi = torch.arange(inner * n, device="cuda", dtype=torch.float32).reshape(inner, n) % 4093
    pick = torch.zeros(edges, n, device="cuda")
    pick[torch.arange(edges), (torch.arange(edges) * 7) % n] = 1.0
    (picked,) = torch.autograd.grad(radial_linear(h, wi), (h,), pick)
    assert torch.equal(picked, wi.t()[(torch.arange(edges, device="cuda") * 7) % n])


@pytest.mark.parametrize("inner", [64, 128])
@pytest.mark.parametrize("edges,n", [(63, 64), (65, 32), (300, 2944), (3000, 544)])
@pytest.mark.parametrize("largest", ["first", "last", "anywhere"])
def test_scales_of_the_split_products_follow_the_terms(inner, edges, n, largest):
    """Operands whose magnitude differs by up to 2^40 from row to row and along the sums: every result
    within float32 rounding of its own sum of magnitudes (2^-24 a term for the split operands and for the
    sums, as for operands of one size)."""
    g = torch.Generator(device="cuda").manual_seed(inner + edges + n)

    def spread(count):
        e = torch.linspace(-20, 20, count, device="cuda").round()
        if largest == "first":
            e = e.flip(0)
        if largest == "anywhere":
            e = e[torch.randperm(count, device="cuda", generator=g)]
        return torch.exp2(e)

    h = (torch.randn(edges, inner, device="cuda", generator=g) * spread(edges)[:, None]
         * spread(inner)[None]).requires_grad_(True)
    w = (torch.randn(inner, n, device="cuda", generator=g) * spread(n)[None]).requires_grad_(True)
    ds = torch.randn(edges, n, device="cuda", generator=g) * spread(edges)[:, None] * spread(n)[None]
    ds[edges // 2] = 0.0
    s = radial_linear(h, w)
    dh, dw = torch.autograd.grad(s, (h, w), ds)
    hd, wd, dd = h.detach().double(), w.detach().double(), ds.double()
    for got, a, b, terms in ((s.detach(), hd, wd, inner), (dh, dd, wd.t().contiguous(), n),
                             (dw, hd.t().contiguous(), dd, edges)):
        bound = (8 + terms ** 0.5) * 2.0 ** -24 * (a.abs() @ b.abs())
        assert bool(((got.double() - a @ b).abs() <= bound).all())


def _assert_products(h, w, ds):
    """s, dh and dw within the bound of `test_scales_of_the_split_products_follow_the_terms`."""
    h, w = h.requires_grad_(True), w.requires_grad_(True)
    s = radial_linear(h, w)
    dh, dw = torch.autograd.grad(s, (h, w), ds)
    hd, wd, dd = h.detach().double(), w.detach().double(), ds.double()
    for name, got, a, b, terms in (("s", s.detach(), hd, wd, h.shape[1]), ("dh", dh, dd, wd.t().contiguous(), w.shape[1]),
                                   ("dw", dw, hd.t().contiguous(), dd, h.shape[0])):
        over = (got.double() - a @ b).abs() / ((8 + terms ** 0.5) * 2.0 ** -24 * (a.abs() @ b.abs())).clamp_min(1e-300)
        assert float(over.max()) <= 1.0, (name, float(over.max()))


@pytest.mark.parametrize("inner", [64, 128])
@pytest.mark.parametrize("edges,n", [(65, 32), (300, 2944), (3000, 544)])
@pytest.mark.parametrize("bits", [8, 14, 20, 40])
def test_spreads_that_oppose_each_other(inner, edges, n, bits):
    """Along each of the three sums one operand grows where the other shrinks, so that all terms are of a size: a small
    operand of a row is not lost beside a large one."""
    g = torch.Generator(device="cuda").manual_seed(inner + edges + n + bits)

    def spread(count):
        return torch.exp2(torch.randint(-bits, bits + 1, (count,), device="cuda", generator=g).float())

    over_edges, over_inner, over_n = spread(edges)[:, None], spread(inner), spread(n)[None]
    h = torch.randn(edges, inner, device="cuda", generator=g) * over_edges * over_inner[None]
    w = torch.randn(inner, n, device="cuda", generator=g) / over_inner[:, None] / over_n
    _assert_products(h, w, torch.randn(edges, n, device="cuda", generator=g) * over_n / over_edges)


@pytest.mark.parametrize("inner", [64, 128])
@pytest.mark.parametrize("outlier", [1e8, 1e10, 1e15])
def test_outliers_that_meet_zeros(inner, outlier):
    """A masked edge whose hidden units hold anything, a unit whose weights are zeros, a column without weights, and
    columns that pick one unit each: the other terms of their sums keep their digits."""
    g = torch.Generator(device="cuda").manual_seed(inner)
    h, w = torch.randn(300, inner, device="cuda", generator=g), torch.randn(inner, 544, device="cuda", generator=g)
    ds = torch.randn(300, 544, device="cuda", generator=g)
    h[17] *= outlier
    ds[17] = 0.0
    h[:, 9] *= outlier
    w[9] = 0.0
    ds[:, 40] *= outlier
    w[:, 40] = 0.0
    picks = torch.arange(64, 64 + 32, device="cuda")
    w[:, picks] = 0.0
    w[10 + torch.arange(32, device="cuda"), picks] = torch.randn(32, device="cuda", generator=g)
    _assert_products(h, w, ds)


@pytest.mark.parametrize("inner,n", [(64, 2944), (64, 96), (128, 1472), (128, 32)])
def test_errors_of_sums_of_one_size(inner, n):
    """Normal values: a sum of k parts of random sign, rounded (or cut off) after each, is 2^-24 sqrt((k + 1) / 2) off, rms,
    beside the rounding of the parts; s adds the upper products of inner / 16 blocks, dh the sums of n / 32 chunks."""
    g = torch.Generator(device="cuda").manual_seed(inner + n)
    h, w = (torch.randn(*shape, device="cuda", generator=g).requires_grad_(True) for shape in ((3001, inner), (inner, n)))
    s = radial_linear(h, w)
    ds = torch.randn(*s.shape, device="cuda", generator=g)
    (dh,) = torch.autograd.grad(s, h, ds)
    h, w, s = h.detach().double(), w.detach().double(), s.detach()
    for name, got, want, parts in (("s", s, h @ w, inner // 16), ("dh", dh, ds.double() @ w.t().contiguous(), n // 32)):
        error = float(((got.double() - want).square().mean() / want.square().mean()).sqrt())
        assert error <= 2.0 ** -24 * ((parts + 1) / 2 + 1) ** 0.5, (name, error)


@pytest.mark.parametrize("inner", [64, 128])
def test_errors_of_the_weight_gradient_have_no_sign(inner):
    """Sums on the matrix cores err downwards: the errors of dW, which is a sum over all edges, do not all have that sign
    (errors of either sign would have a mean of a hundredth of their rms over so many values)."""
    edges, n = 100003, 512
    g = torch.Generator(device="cuda").manual_seed(inner)
    h = torch.nn.functional.silu(torch.randn(edges, inner, device="cuda", generator=g))
    w = torch.randn(inner, n, device="cuda", generator=g).requires_grad_(True)
    ds = torch.randn(edges, n, device="cuda", generator=g)
    (dw,) = torch.autograd.grad(radial_linear(h, w), w, ds)
    error = dw.double() - h.double().t().contiguous() @ ds.double()
    assert abs(float(error.mean())) <= float(error.square().mean().sqrt()) / 8


@pytest.mark.parametrize("inner", [8, 32, 64, 128])
@pytest.mark.parametrize("edges,n", [(5, 2944), (256, 992), (16400, 96), (33000, 736), (33000, 800), (65000, 768), (70000, 64)])
def test_forward_over_ranges_of_columns(inner, edges, n):
    """Few edges: blocks share the columns, an odd number of tiles too; many: each takes all of them."""
    g = torch.Generator(device="cuda").manual_seed(inner + edges)
    h = torch.randn(edges, inner, device="cuda", generator=g)
    w = torch.randn(inner, n, device="cuda", generator=g)
    want = h.double() @ w.double()
    bound = 8 * 2.0 ** -24 * (h.double().abs() @ w.double().abs())
    assert bool(((radial_linear(h, w).double() - want).abs() <= bound).all())


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_a_value_that_is_no_number_stays_in_its_row_and_column(bad):
    g = torch.Generator(device="cuda").manual_seed(3)
    h = torch.randn(300, 64, device="cuda", generator=g)
    w = torch.randn(64, 96, device="cuda", generator=g)
    ds = torch.randn(300, 96, device="cuda", generator=g)
    h[7, 5], ds[200, 40] = bad, bad
    h.requires_grad_(True)
    w.requires_grad_(True)
    s = radial_linear(h, w)
    dh, dw = torch.autograd.grad(s, (h, w), ds)
    rows = lambda t: torch.nonzero(~t.isfinite().all(1)).flatten().tolist()   # noqa: E731
    assert rows(s) == [7] and rows(dh) == [200]
    assert rows(dw[:, torch.arange(96, device="cuda") != 40]) == [5]
    assert not bool(dw[:, 40].isfinite().any())
