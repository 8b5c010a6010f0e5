"""The 32-bit matrix-core products against 64-bit sums: at the edges of their tiles, of K's blocks and parts, with rows a
stride apart, bias and residual, and the operands that they leave to the plain kernels."""

import pytest
import torch

from tokasaurus_amd.kernels import ops
from tokasaurus_amd.kernels.library import load

pytestmark = pytest.mark.gpu


def check(got, a, w, bias=None, residual=None):
    """Every sum of K products and up to two more terms, each rounded: (K + 2) 2^-24 of the sum of the magnitudes."""
    a, w = a.double(), w.double()
    want, size = a @ w.T, a.abs() @ w.abs().T
    for t in (bias, residual):
        if t is not None:
            want, size = want + t.double(), size + t.double().abs()
    worst = ((got.double() - want).abs() / (size + 1e-30)).max()
    assert float(worst) <= (a.shape[1] + 2) * 2.0 ** -24, float(worst)


# tokens at the edges of the few-row kernel (16), of tiles of 32, 64 and 128 tokens; columns and K at the edges of blocks
@pytest.mark.parametrize("m", [1, 4, 15, 16, 17, 32, 33, 64, 65, 129, 300])
@pytest.mark.parametrize("nk", [(1, 4), (4, 12), (18, 16), (63, 36), (64, 260), (77, 512), (260, 516), (1000, 2052), (1133, 1008), (1008, 276)])
def test_sizes(m, nk):
    n, k = nk
    g = torch.Generator(device="cuda").manual_seed(m * 1000 + n + k)
    wide = torch.randn((m, k + 8), generator=g, device="cuda")
    a = wide[:, 4 : k + 4]  # rows a stride apart, 16-byte aligned
    w = torch.randn((n, k), generator=g, device="cuda")
    bias = torch.randn((n,), generator=g, device="cuda")
    residual = torch.randn((m, n + 3), generator=g, device="cuda")[:, 1 : n + 1]
    assert load("core").tk_gemm_f32_takes(a.data_ptr(), a.stride(0), w.data_ptr(), k) == 1
    check(ops.gemm_generic(a, w), a, w)
    check(ops.gemm_generic(a, w, residual=residual, bias=bias), a, w, bias, residual)


@pytest.mark.parametrize("m", [1, 7, 8, 9])
@pytest.mark.parametrize("nk", [(1, 256), (8, 288), (20, 4096), (2047, 320), (2048, 2080), (2049, 256)])
def test_few_rows_by_halves_of_k(m, nk):
    """Weights of few enough rows for 8 a workgroup: neighbouring blocks of K beside each other, with blocks left over, and the sizes around."""
    n, k = nk
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a, w = torch.randn((m, k + 4), generator=g, device="cuda")[:, 4:], torch.randn((n, k), generator=g, device="cuda")
    bias, residual = torch.randn((n,), generator=g, device="cuda"), torch.randn((m, n + 3), generator=g, device="cuda")[:, 1 : n + 1]
    check(ops.gemm_generic(a, w), a, w)
    check(ops.gemm_generic(a, w, residual=residual, bias=bias), a, w, bias, residual)


def test_large_tiles():
    g = torch.Generator(device="cuda").manual_seed(5)
    a = torch.randn((2100, 100), generator=g, device="cuda")
    w = torch.randn((4104, 100), generator=g, device="cuda")  # 17 x 33 tiles of 128 x 128
    check(ops.gemm_generic(a, w), a, w)


@pytest.mark.parametrize("m", [3, 40])
@pytest.mark.parametrize("shape", ["odd inner size", "odd start", "odd stride"])
def test_operands_left_to_the_plain_kernels(m, shape):
    g = torch.Generator(device="cuda").manual_seed(m)
    k = 50 if shape == "odd inner size" else 52
    wide = torch.randn((m, k + (9 if shape == "odd stride" else 8)), generator=g, device="cuda")
    a = wide[:, 1 : k + 1] if shape == "odd start" else wide[:, :k]
    w = torch.randn((70, k), generator=g, device="cuda")
    assert load("core").tk_gemm_f32_takes(a.data_ptr(), a.stride(0), w.data_ptr(), k) == 0
    check(ops.gemm_generic(a, w), a, w)


@pytest.mark.parametrize("m", [2, 20, 70])
def test_infinities_and_nan_stay_in_their_rows(m):
    g = torch.Generator(device="cuda").manual_seed(m)
    a = torch.randn((m, 64), generator=g, device="cuda")
    w = torch.randn((40, 64), generator=g, device="cuda").abs() + 0.1
    a[0, 3], a[1, 5] = float("inf"), float("nan")
    got = ops.gemm_generic(a, w)
    assert torch.isinf(got[0]).all() and torch.isnan(got[1]).all() and torch.isfinite(got[2:]).all()


@pytest.mark.parametrize("m", [17, 32, 33, 64, 65, 129, 300])
@pytest.mark.parametrize("nk", [(1, 32), (63, 64), (64, 96), (260, 128), (1000, 160), (1133, 1024), (2052, 992)])
def test_steps_straight_to_local_memory(m, nk):
    """Inner sizes of whole steps: fewer than local memory holds, as many, and more; every one in one and in several parts."""
    test_sizes(m, nk)


def test_largest_tiles_straight_to_local_memory():
    """128 x 128, which take as many tiles as fill the chip twice; rows and columns that end inside one."""
    for m, n, k in ((2100, 4100, 64), (2048, 4160, 96), (2049, 4096, 32)):
        test_sizes(m, (n, k))


@pytest.mark.parametrize("m", [1, 3, 4, 8])
@pytest.mark.parametrize("nk", [(20, 8192), (9, 8224), (2050, 8192), (24, 16384)])
def test_few_rows_over_long_inner_sizes(m, nk):
    """Where a wavefront has several sets of loads, and workgroups begin at different ones."""
    test_sizes(m, nk)


@pytest.mark.parametrize("nk", [(2048, 8192), (1031, 8192), (77, 16384), (300, 9248), (2048, 2048), (70, 256)])
def test_a_rows_bits_do_not_depend_on_how_many_rows_there_are(nk):
    """Steps of up to 8 rows are recorded with 1, 2, 4 or 8: a row alone, among 3 and among the recorded sizes is the same sums in one order."""
    n, k = nk
    g = torch.Generator(device="cuda").manual_seed(n + k)
    a, w = torch.randn((8, k), generator=g, device="cuda"), torch.randn((n, k), generator=g, device="cuda")
    all_rows = ops.gemm_generic(a, w)
    for m in range(1, 8):
        assert torch.equal(ops.gemm_generic(a[:m], w), all_rows[:m]), m
