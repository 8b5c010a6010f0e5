"""Products of many rows in tiles: every tile, rows and outputs that end inside one, as many steps of K as local memory holds and
fewer and more, rows a stride apart, the plain and the gated form, against sums in 64-bit."""

from __future__ import annotations

import pytest
import torch

from test_glu_stream_gpu import _case, _check, _silu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", range(5))
@pytest.mark.parametrize("m", [1, 127, 200, 577])
@pytest.mark.parametrize("n,k", [(8, 64), (136, 128), (72, 192), (520, 256), (1000, 320), (264, 448), (1288, 1024)])
def test_against_64_bit_sums(shape, m, n, k):
    from tokasaurus_amd.kernels import ops

    x, w, _ = _case(m, n, k, 7 * m + n + k + shape)
    wide = torch.zeros((m, k + 8), dtype=torch.bfloat16)  # rows apart
    wide[:, :k] = x
    rows = wide.cuda()[:, :k]
    _check(ops.gemm_tiles_bf16(rows, w.cuda(), shape, glu=True), x.double(), w, _silu, k)
    if shape >= 3:
        return  # gated only
    plain = ops.gemm_tiles_bf16(rows, w.cuda(), shape)
    want, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    # 32-bit sums of k products (k 2^-24 of their sizes), rounded once to bfloat16 (8 bits: 2^-8 of the value at most)
    assert ((plain.cpu().double() - want).abs() <= want.abs() * 2.0 ** -8 + size * (k + 8) * 2.0 ** -23).all()


@pytest.mark.parametrize("m", [1, 65, 127, 128, 129, 300])
@pytest.mark.parametrize("n,k", [(8, 64), (32, 128), (72, 320), (520, 384), (1000, 448), (264, 1024)])
def test_gated_tiles_of_64_weight_rows(m, n, k):
    """Fewer steps of K than local memory holds, as many and more; outputs that end inside a tile of 32."""
    from tokasaurus_amd.kernels import ops

    x, w, _ = _case(m, n, k, 3 * m + n + k)
    wide = torch.zeros((m, k + 8), dtype=torch.bfloat16)  # rows apart
    wide[:, :k] = x
    _check(ops.gemm_tiles_bf16(wide.cuda()[:, :k], w.cuda(), 5, glu=True), x.double(), w, _silu, k)


@pytest.mark.parametrize("m,n,k,glu", [(65, 8192, 2048, True), (101, 8192, 2048, True), (1000, 2048, 1024, True), (1270, 3072, 512, False), (1800, 2048, 192, False)])
def test_linear_takes_them(monkeypatch, m, n, k, glu):
    """The rule's tiles through the linear map."""
    from tokasaurus_amd.kernels import ops
    from tokasaurus_amd.parts.linear import Linear

    made, call = [], ops.call
    monkeypatch.setattr(ops, "call", lambda name, *a: made.append(name) or call(name, *a))

    assert ops.tiles_choice(m, n, k, glu) >= 0 and ops.tiles_choice(m, n, k - 8, glu) == -1
    x, w, gen = _case(m, n, k, m + n)
    w = w if glu else w[:n]
    lin = Linear(k, ["w"], [w.shape[0]])
    lin.weight = w.cuda()
    if glu:
        _check(lin(x.cuda(), swiglu=True), x.double(), w, _silu, k)
        assert made == ["tk_gemm_tiles_bf16"]
        return
    res = torch.randn((m, n), generator=gen).bfloat16()
    prod = x.double() @ w.double().t()
    want = prod + res.double()
    got = lin(x.cuda(), residual=res.cuda()).cpu().double()
    assert made == ["tk_gemm_tiles_bf16", "tk_add"]
    # the product rounded (2^-8 of it at most), then the sum; 32-bit sums of products of size 1 / sqrt(k), a few of them
    assert ((got - want).abs() <= (want.abs() + 1.01 * prod.abs()) * 2.0 ** -8 + 1e-4).all()


def test_refused():
    from tokasaurus_amd.kernels import ops
    from tokasaurus_amd.kernels.library import KernelError

    x, w, _ = _case(200, 64, 128, 1)
    for bad in (lambda: ops.gemm_tiles_bf16(x.cuda()[:, :96], w.cuda()[:, :96].contiguous(), 0),  # a step of K cut short
                lambda: ops.gemm_tiles_bf16(x.cuda(), w.cuda(), 5), lambda: ops.gemm_tiles_bf16(x.cuda(), w.cuda(), 3),
                lambda: ops.gemm_tiles_bf16(x.cuda(), w.cuda(), 6, glu=True), lambda: ops.gemm_tiles_bf16(x.cuda()[:, 4:68], w.cuda()[:, :64].contiguous(), 0)):
        with pytest.raises(KernelError):
            bad()
