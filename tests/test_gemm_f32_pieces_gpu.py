"""32-bit products of many rows by exact pieces of the numbers: against 64-bit sums and against the unsplit products (which an inner size of
no whole steps goes to), at the edges of both tiles and of K's parts, with numbers at the ends of their range."""

import pytest
import torch

from tokasaurus_amd.kernels import ops
from tokasaurus_amd.kernels.library import load

pytestmark = pytest.mark.gpu


def unsplit(a, w, **more):
    pad = lambda x: torch.nn.functional.pad(x, (0, 4))  # noqa: E731
    return ops.gemm_generic(pad(a), pad(w), **more)


def error(got, want):
    return float((got.double() - want).norm() / want.norm())


# (rows counted in tiles of 64) x columns x K at 7 * 2^27 and over; columns that no 16 bytes hold (K in one part), K of one step of parts and of many
@pytest.mark.parametrize("m,n,k", [(33, 14336, 1024), (64, 14337, 1024), (65, 7170, 1056), (129, 4780, 1024), (300, 1233, 2400), (65, 820, 9088), (1000, 3588, 256),
                                   (2049, 1604, 288), (512, 2400, 768), (1025, 4100, 512)])
def test_errors_are_no_larger_than_unsplit(m, n, k):
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    wide = torch.randn((m, k + 8), generator=g, device="cuda")
    a, w = wide[:, 4 : k + 4], torch.randn((n, k), generator=g, device="cuda")  # rows a stride apart
    bias, residual = torch.randn((n,), generator=g, device="cuda"), torch.randn((m, n + 3), generator=g, device="cuda")[:, 1 : n + 1]
    want, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    got = ops.gemm_generic(a, w)
    # a sum of K products, each rounded, and what is left of each product (2^-30 at most)
    assert bool(((got.double() - want).abs() <= ((k + 2) * 2.0 ** -24 + 2.0 ** -30) * size).all())
    assert error(got, want) <= error(unsplit(a, w), want)
    want = want + bias.double() + residual.double()
    assert error(ops.gemm_generic(a, w, bias=bias, residual=residual), want) <= error(unsplit(a, w, bias=bias, residual=residual), want) * 1.01


# a tile of 64 rows and one of 128, K in one part each (a part of a row without terms is a sum of zero, and made unsplit)
@pytest.mark.parametrize("m,n,k", [(33, 28672, 512), (2048, 2048, 2048)])
@pytest.mark.parametrize("terms", [1, 2, 3, 5, 8, 16, 40])
def test_few_terms_a_row(m, n, k, terms):
    """Ordinary numbers, the row with all bits of its numbers set among them, element by element."""
    assert load("core").tk_gemm_f32_cuts(m, n, k) == 1
    g = torch.Generator(device="cuda").manual_seed(m + terms)
    a, w = torch.zeros((m, k), device="cuda"), torch.randn((n, k), generator=g, device="cuda")
    at = torch.rand((m, k), generator=g, device="cuda").topk(terms, -1).indices
    a.scatter_(1, at, torch.randn((m, terms), generator=g, device="cuda"))
    a[0] = a[0].sign() * (1 + 2.0 ** -7 - 2.0 ** -23)
    w[:100] = w[:100].sign() * (1 + 2.0 ** -7 - 2.0 ** -23)
    want, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    got = ops.gemm_generic(a, w)
    # the greatest pieces' product is exact; each further one is added with a rounding (by truncation at worst), the others once, at the end;
    # what is left of a product is under 2^-30
    assert bool(((got.double() - want).abs() <= ((2 * terms - 1) * 2.0 ** -24 + 2.0 ** -29) * size).all())
    assert error(got, want) <= error(unsplit(a, w), want) * (1.01 if terms == 1 else 1)


@pytest.mark.parametrize("m", [70, 300])
def test_numbers_at_the_ends_of_their_range(m):
    g = torch.Generator(device="cuda").manual_seed(m)
    n, k = 7300, 1024
    a, w = torch.randn((m, k), generator=g, device="cuda"), torch.randn((n, k), generator=g, device="cuda").abs() + 0.1
    a[0, 3], a[1, 5], a[2, 7] = float("inf"), float("nan"), -float("inf")
    a[3] *= 2.0 ** -130
    a[4] = 0
    a[5] *= 2.0 ** 112
    a[6, 1:] = 0
    a[6, 0] = 2.0 ** -140
    got = ops.gemm_generic(a, w)
    assert bool((got[0] == float("inf")).all() and torch.isnan(got[1]).all() and (got[2] == -float("inf")).all())
    assert bool(torch.isfinite(got[3:]).all()) and bool((got[4] == 0).all())
    want = a[3:].double() @ w.double().T
    for i in (0, 2):
        assert error(got[3 + i], want[i]) <= 2e-6, i
    # one product of a number below the least normal one: rounded to a multiple of 2^-149
    assert bool(((got[6].double() - want[3]).abs() <= 2.0 ** -149).all())
    assert error(got[7:], want[4:]) <= 2e-6


@pytest.mark.parametrize("m", [70, 300])
@pytest.mark.parametrize("down,up", [(-118, 110), (110, -118), (-140, 127), (0, 40)])
def test_numbers_whose_pieces_are_lost(m, down, up):
    """Small numbers beside large ones: what their pieces leave out would be the whole of an ordinary sum."""
    g = torch.Generator(device="cuda").manual_seed(m + up)
    n, k = 7300, 1024
    a, w = (torch.rand((r, k), generator=g, device="cuda") + 0.5 for r in (m, n))
    a, w = (torch.ldexp(torch.ldexp(x, torch.tensor(e // 2, device="cuda")), torch.tensor(e - e // 2, device="cuda")) for x, e in ((a, down), (w, up)))
    got, want = ops.gemm_generic(a, w), a.double() @ w.double().T
    assert error(got, want) <= 2e-6
    a[:, 1:] = 0  # one product a sum
    got, want = ops.gemm_generic(a, w), a.double() @ w.double().T
    assert bool(((got.double() - want).abs() <= 2.0 ** -24 * want.abs()).all())


def test_more_rows_than_a_grid_has():
    g = torch.Generator(device="cuda").manual_seed(2)
    m, n, k = 65568, 16, 1024
    a, w = torch.randn((m, k), generator=g, device="cuda"), torch.randn((n, k), generator=g, device="cuda")
    residual = torch.randn((m, n), generator=g, device="cuda")
    assert error(ops.gemm_generic(a, w, residual=residual), a.double() @ w.double().T + residual.double()) <= 1e-6


# tiles of 64 and of 128 rows, K in one part and in several, columns that no 16 bytes hold
@pytest.mark.parametrize("m,n,k,cuts", [(33, 28672, 512, False), (70, 7300, 1024, True), (2048, 2048, 2048, False), (300, 7300, 1024, True), (65, 7170, 1056, False)])
def test_a_row_changes_no_other_row(m, n, k, cuts):
    """Zeros, numbers without pieces, very large ones, infinity and NaN in a row of either operand: the bits of all results that are not made of it
    stay, and its own are right."""
    assert (load("core").tk_gemm_f32_cuts(m, n, k) > 1) == cuts
    g = torch.Generator(device="cuda").manual_seed(m)
    a, w = torch.randn((m, k), generator=g, device="cuda"), torch.randn((n, k), generator=g, device="cuda")
    residual = torch.randn((m, n), generator=g, device="cuda")
    before = ops.gemm_generic(a, w, residual=residual)
    odd = [torch.zeros(k), torch.randn(k) * 2.0 ** -118, torch.randn(k) * 2.0 ** 31, torch.randn(k) * 2.0 ** 60, torch.full((k,), float("nan")),
           torch.randn(k).scatter(0, torch.tensor([k - 1]), float("inf")), torch.randn(k).scatter(0, torch.tensor([3]), 2.0 ** 40)]
    for row in odd:
        for side, at in (("a", m // 2), ("w", n - 3)):
            x, y = a.clone(), w.clone()
            (x if side == "a" else y)[at] = row.cuda()
            got = ops.gemm_generic(x, y, residual=residual)
            rest = lambda t: torch.cat([t[:at], t[at + 1:]]) if side == "a" else torch.cat([t[:, :at], t[:, at + 1:]], 1)  # noqa: E731
            assert torch.equal(rest(got), rest(before))
            own = got[at].double() if side == "a" else got[:, at].double()
            other, beside = (w, residual[at]) if side == "a" else (a, residual[:, at])
            want = other.double() @ row.cuda().double() + beside.double()
            if bool(torch.isfinite(row).all()):
                assert bool(((own - want).abs() <= (k + 2) * 2.0 ** -24 * (other.double().abs() @ row.cuda().double().abs() + beside.double().abs())).all())
            else:
                assert torch.equal(own.isnan(), want.isnan()) and torch.equal(own[~own.isnan()], want[~want.isnan()])


def test_many_products_whose_pieces_lose_a_little():
    """65,536 numbers of 2^-125 beside some of up to 2^39 and one product of 2^-59 behind them: what their pieces lose is little of a product and 2^-20 of the sum."""
    g = torch.Generator(device="cuda").manual_seed(4)
    m, n, k = 64, 901, 65536
    assert load("core").tk_gemm_f32_cuts(m, n, k) == 1
    a = (torch.rand((m, k), generator=g, device="cuda") + 1) * 2.0 ** -125
    w = (torch.rand((n, k), generator=g, device="cuda") + 1) * 2.0 ** 38
    a[:, -1], w[:, -1] = 2.0 ** -60, 2.0
    got, want = ops.gemm_generic(a, w), a.double() @ w.double().T
    # one rounding, and up to 31 of the small products added behind the great one, each below half a place of it
    assert bool(((got.double() - want).abs() <= (2.0 ** -24 + 31 * 2.0 ** (-86 + 1.2 + 59)) * want).all())
