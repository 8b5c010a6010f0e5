"""Gate and up for up to 64 rows through local memory: every number of rows and steps where the kernel's ring of steps fills,
wraps and drains, ragged widths, the norm in front and what follows, against sums in 64-bit."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(m, n, k, seed):
    gen = torch.Generator().manual_seed(seed)
    return (torch.randn((m, k), generator=gen).bfloat16(), (torch.randn((2 * n, k), generator=gen) / k ** 0.5).bfloat16(), gen)


def _check(out, x64, w, act, k, bias=None):
    """Gate and up are 32-bit sums of k products (error k 2^-24 of the products' sizes, and again for the scaling), rounded to
    bfloat16 (2^-8) before the activation, whose slope is below 1.1 in the gate; the result is rounded again."""
    n = w.shape[0] // 2
    p = x64 @ w.double().t()
    size = x64.abs() @ w.double().abs().t()
    if bias is not None:
        p = p + bias.double()
    g, u = p[:, :n], p[:, n:]
    eg, eu = (t.abs() * 2.0 ** -8 + s * (k + 8) * 2.0 ** -23 for t, s in ((g, size[:, :n]), (u, size[:, n:])))
    want, reach = act(g, u)
    limit = want.abs() * 2.0 ** -7.5 + 1.2 * (u.abs() + 1 + eu) * eg + reach * eu + 1e-6
    assert ((out.cpu().double() - want).abs() <= limit).all()


def _silu(g, u):
    return torch.nn.functional.silu(g) * u, torch.nn.functional.silu(g).abs() + 1e-3


@pytest.mark.parametrize("m", [1, 2, 16, 17, 32, 33, 47, 64])
@pytest.mark.parametrize("n,k", [(32, 64), (40, 192), (1000, 256), (33, 320), (8, 384), (96, 448), (4100, 2048)])
def test_against_64_bit_sums(m, n, k):
    from tokasaurus_amd.kernels import ops

    x, w, _ = _case(m, n, k, 7 * m + n + k)
    out = ops.gemm_skinny_bf16(x.cuda(), w.cuda(), swiglu=True, staged=2)
    _check(out, x.double(), w, _silu, k)


@pytest.mark.parametrize("m", [3, 30, 64])
def test_norm_in_front_bias_and_other_activations(m):
    from tokasaurus_amd.kernels import ops

    n, k = 72, 512
    x, w, gen = _case(m, n, k, m)
    wide = torch.zeros((m, k + 64), dtype=torch.bfloat16)  # rows apart
    wide[:, :k] = x
    bias = torch.randn((2 * n,), generator=gen).bfloat16()
    out = ops.gemm_skinny_bf16(wide.cuda()[:, :k], w.cuda(), swiglu=True, staged=2, bias=bias.cuda())
    _check(out, x.double(), w, _silu, k, bias)
    gelu = lambda g, u: (torch.nn.functional.gelu(g, approximate="tanh") * u, torch.nn.functional.gelu(g, approximate="tanh").abs() + 1e-3)
    _check(ops.gemm_skinny_bf16(x.cuda(), w.cuda(), swiglu=True, staged=2, glu="gelu_tanh"), x.double(), w, gelu, k)
    for parts in (5, 8):
        sumsq = torch.rand((m, parts), generator=gen) * k / parts
        pre = ops.Prenorm(x.cuda(), sumsq.cuda())
        out = ops.gemm_skinny_bf16(pre.scaled, w.cuda(), swiglu=True, staged=2, prenorm=pre, norm_eps=1e-5)
        rows = x.double() / torch.sqrt(sumsq.double().sum(1, keepdim=True) / k + 1e-5)
        _check(out, rows, w, _silu, k)


@pytest.mark.parametrize("m,n,k,streamed", [(2, 8192, 3072, True), (1, 8192, 3072, True), (16, 8192, 2048, True), (1, 8192, 2048, True),
                                            (1, 8224, 4096, False), (2, 8224, 4096, True), (1, 12320, 4096, True), (1, 8160, 4096, False),
                                            (20, 4096, 2048, True), (17, 4096, 2048, True), (16, 4096, 2048, False), (64, 1000, 1024, True),
                                            (20, 512, 2080, False)])
def test_which_calls_are_streamed(m, n, k, streamed):
    """The streamed form and the weight-streaming one differ in their order of summation, hence in some results.  Streamed are as many
    outputs as give every compute unit a workgroup from one row on, fewer from 40,000 elements of x on (counted at the
    recorded size, 32 for 17 rows); not one row of a long inner size where few units have a second workgroup."""
    from tokasaurus_amd.kernels import ops

    x, w, _ = _case(m, n, k, m + k)
    x, w = x.cuda(), w.cuda()
    chosen = ops.gemm_skinny_bf16(x, w, swiglu=True)
    if k % 64:
        with pytest.raises(Exception, match="multiple of 64"):
            ops.gemm_skinny_bf16(x, w, swiglu=True, staged=2)
    else:
        assert torch.equal(chosen, ops.gemm_skinny_bf16(x, w, swiglu=True, staged=2)) == streamed
    assert torch.equal(chosen, ops.gemm_skinny_bf16(x, w, swiglu=True, staged=0)) != streamed


def test_rows_of_gate_and_up():
    from tokasaurus_amd.kernels import ops

    assert ops.glu_rows(2048) == ops.glu_rows(64) == 64 and ops.glu_rows(2080) == ops.skinny_rows(2080, paired=True)


@pytest.mark.parametrize("m", [20, 40, 64])
@pytest.mark.parametrize("layout", ["odd stride", "odd start", "columns"])
def test_rows_that_lie_anywhere_take_the_librarys_product(m, layout):
    """Rows of 20 and more were the library's, which reads them wherever they lie."""
    from tokasaurus_amd.kernels import ops
    from tokasaurus_amd.parts.linear import Linear

    n, k = 72, 4096
    x, w, _ = _case(m, n, k, m)
    buf = torch.zeros((m, k + 9), dtype=torch.bfloat16, device="cuda")
    rows = {"odd stride": buf[:, :k], "odd start": buf.view(-1)[1 : 1 + m * k].view(m, k), "columns": buf.view(-1)[: m * k].view(k, m).t()}[layout]
    rows.copy_(x)
    lin = Linear(k, ["gate", "up"], [n, n])
    lin.weight = w.cuda()
    assert ops.skinny_rows(k, paired=True) < m <= ops.glu_rows(k, n) and not ops.rows_at_16_bytes(rows)
    _check(lin(rows, swiglu=True), x.double(), w, _silu, k)
