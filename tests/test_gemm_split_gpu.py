"""Products with K cut among workgroups and the passes that add the cuts, at the edges of the kernel's blocks of rows, tiles of
weight rows and ring of steps, against sums in 64-bit and against the passes behind a whole product."""

from __future__ import annotations

import pytest
import torch

from tokasaurus_amd.kernels import ops
from tokasaurus_amd.kernels.library import call

pytestmark = pytest.mark.gpu


def _case(m, n, k, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    wide = torch.randn((m, k + 64), generator=gen, device="cuda").bfloat16()
    return wide[:, 32 : k + 32], (torch.randn((n, k), generator=gen, device="cuda") / k ** 0.5).bfloat16(), gen


@pytest.mark.parametrize("m", [1, 15, 16, 17, 32, 33, 64, 65, 96, 97, 128, 129, 200, 256])
@pytest.mark.parametrize("n,k", [(8, 64), (72, 192), (64, 256), (200, 1088), (2048, 2048), (3000, 960)])
def test_cuts_against_64_bit_sums(m, n, k):
    """Every cut is 32-bit sums of at most k products, and their sum has as many terms as there are cuts: (k + 16) 2^-24 of the
    sum of the magnitudes."""
    x, w, _ = _case(m, n, k, m + n + k)
    want, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    part = ops.gemm_split(x, w)
    assert part.shape == (ops.split_cuts(n, k, m), m, n)
    for cuts in {1, 2, 3, k // 64}:
        if cuts > k // 64:
            continue
        own = torch.full((cuts, m, n), float("nan"), device="cuda")
        call("tk_gemm_split_bf16", x.data_ptr(), x.stride(0), w.data_ptr(), own.data_ptr(), m, n, k, cuts, torch.cuda.current_stream().cuda_stream)
        for got in (part, own):
            assert float(((got.double().sum(0) - want).abs() / (size + 1e-30)).max()) <= (k + 16) * 2.0 ** -24


@pytest.mark.parametrize("rows,hidden,cuts", [(1, 8, 1), (3, 72, 5), (17, 2048, 8), (5, 4096, 4), (2, 8192, 3), (2, 9000, 2)])
@pytest.mark.parametrize("w32", [False, True])
def test_residual_sum_and_norm(rows, hidden, cuts, w32):
    """The very bits of the pass behind a whole product, for a product that is the cuts' sum in ascending order."""
    gen = torch.Generator(device="cuda").manual_seed(hidden + cuts)
    part = torch.randn((cuts, rows, hidden), generator=gen, device="cuda")
    residual = torch.randn((rows, hidden), generator=gen, device="cuda").bfloat16()
    weight = torch.randn((hidden,), generator=gen, device="cuda")
    weight = weight if w32 else weight.bfloat16()
    whole = part[0].clone()
    for c in range(1, cuts):
        whole += part[c]
    for got, want in zip(ops.split_add_rmsnorm(part, residual, weight, 1e-5), ops.add_rmsnorm(whole.bfloat16(), residual, weight, 1e-5)):
        assert torch.equal(got, want)


@pytest.mark.parametrize("rows,hidden,cuts", [(1, 8, 1), (3, 72, 5), (17, 2048, 8), (2, 9000, 2)])
@pytest.mark.parametrize("w32", [False, True])
def test_normed_rows_rounded_once(rows, hidden, cuts, w32):
    """The rows that go on are as without it; the normed ones are their 64-bit norm rounded once (8 significant bits: 2^-8 of the value at
    most, twice rounded up to 2^-7; the sum of squares, its root and the product are 32-bit: well under 2^-15)."""
    gen = torch.Generator(device="cuda").manual_seed(hidden + cuts + 1)
    part, residual = torch.randn((cuts, rows, hidden), generator=gen, device="cuda"), torch.randn((rows, hidden), generator=gen, device="cuda").bfloat16()
    weight = torch.randn((hidden,), generator=gen, device="cuda")
    weight = weight if w32 else weight.bfloat16()
    stream, normed = ops.split_add_rmsnorm(part, residual, weight, 1e-5, once=True)
    assert torch.equal(stream, ops.split_add_rmsnorm(part, residual, weight, 1e-5)[0])
    x = stream.double()
    want = x / torch.sqrt((x * x).mean(1, keepdim=True) + 1e-5) * weight.double()
    assert ((normed.double() - want).abs() <= want.abs() * (2.0 ** -8 + 2.0 ** -15)).all()


@pytest.mark.parametrize("rows,n,k", [(6, 2048, 8192), (24, 2048, 2048), (4, 4096, 14336)])
def test_few_rows_are_rounded_once_behind_a_linear_map(rows, n, k):
    """As many rows as the weight-streaming product would have taken, in the split form: what stands behind the norm is rounded once."""
    from tokasaurus_amd.parts.linear import Linear
    from tokasaurus_amd.parts.norm import RMSNorm

    x, w, gen = _case(rows, n, k, rows + n)
    lin, norm = Linear(k, ["w"], [n]), RMSNorm(n, 1e-5, "n")
    lin.weight, norm.weight = w, (1 + 0.1 * torch.randn((n,), generator=gen, device="cuda")).bfloat16()
    assert lin.split_norm_from <= rows <= ops.skinny_rows(k)
    stream, prepared = lin.with_residual(x, torch.randn((rows, n), generator=gen, device="cuda").bfloat16(), norm)
    s = stream.double()
    want = s / torch.sqrt((s * s).mean(1, keepdim=True) + 1e-5) * norm.weight.double()
    assert ((prepared.normed.double() - want).abs() <= want.abs() * (2.0 ** -8 + 2.0 ** -15)).all()


@pytest.mark.parametrize("nq,nkv,d,page", [(4, 2, 16, 16), (32, 8, 64, 16), (5, 5, 80, 4), (16, 2, 128, 32)])
@pytest.mark.parametrize("tables", [True, False])
def test_rotation_and_append(nq, nkv, d, page, tables):
    rows, cuts, width = 19, 3, (nq + 2 * nkv) * d
    gen = torch.Generator(device="cuda").manual_seed(d)
    part = torch.randn((cuts, rows, width), generator=gen, device="cuda")
    whole = (part[0] + part[1]) + part[2]
    positions = torch.randperm(3 * page, generator=gen, device="cuda")[:rows].to(torch.int32) if 3 * page >= rows else torch.arange(rows, device="cuda", dtype=torch.int32) % (3 * page)
    req = torch.arange(rows, device="cuda", dtype=torch.int32)
    table = torch.randperm(rows * 3, generator=gen, device="cuda").to(torch.int32).view(rows, 3)
    cos, sin = ops.rope_table(1.0 / 10000 ** (torch.arange(0, d, 2, device="cuda").float() / d), 3 * page) if tables else (None, None)
    pages = [[torch.zeros(shape(rows * 3, nkv, page, d), dtype=torch.bfloat16, device="cuda") for shape in (ops.key_pages_shape, ops.value_pages_shape)]
             for _ in range(2)]
    got = ops.split_rope_append(part, ops.RopeAppend(positions, req, table, cos, sin, *pages[0], nq, nkv, d, page))
    stacked = whole.bfloat16()
    ops.rope_append(stacked, positions, req, table, cos, sin, *pages[1], nq, nkv, d, page)
    assert torch.equal(got, stacked[:, : nq * d])
    assert torch.equal(pages[0][0], pages[1][0]) and torch.equal(pages[0][1], pages[1][1])
    assert pages[0][0].count_nonzero() > 0


@pytest.mark.parametrize("n,k", [(2048, 8192), (2048, 2048), (4096, 14336)])
@pytest.mark.parametrize("m,size", [(3, 4), (5, 8), (9, 16), (11, 16), (17, 32), (33, 48), (39, 48), (65, 80), (113, 128)])
def test_a_row_padded_to_a_recorded_size_keeps_its_bits(m, size, n, k):
    """A decode step of m rows alone and padded to the size that it is recorded at: output or down projection with the norm behind
    it, and the stacked q, k, v product, by one kernel, where both counts are few rows or split products."""
    from tokasaurus_amd.parts.linear import Linear
    from tokasaurus_amd.parts.norm import RMSNorm

    x, w, gen = _case(size, n, k, size + n + k)
    lin, norm = Linear(k, ["w"], [n]), RMSNorm(n, 1e-5, "n")
    lin.weight, norm.weight = w, torch.ones((n,), dtype=torch.bfloat16, device="cuda")
    residual = torch.randn((size, n), generator=gen, device="cuda").bfloat16()
    (a, pa), (b, pb) = lin.with_residual(x[:m], residual[:m], norm), lin.with_residual(x, residual, norm)
    assert torch.equal(a, b[:m])
    assert (pa.data is None) == (pb.data is None)
    for p, q in [(pa.normed, pb.normed)] if pa.data is None else [(pa.data.scaled, pb.data.scaled), (pa.data.sumsq, pb.data.sumsq)]:
        assert torch.equal(p, q[:m])


@pytest.mark.parametrize("m,size", [(3, 4), (5, 8), (9, 16), (11, 16), (17, 32), (33, 48), (113, 128)])
def test_rotated_rows_padded_to_a_recorded_size_keep_their_bits(m, size):
    from tokasaurus_amd.parts.linear import Linear

    nq, nkv, d, page = 32, 8, 64, 16
    x, w, gen = _case(size, (nq + 2 * nkv) * d, 2048, size)
    lin = Linear(2048, ["w"], [(nq + 2 * nkv) * d])
    lin.weight = w
    cos, sin = ops.rope_table(1.0 / 10000 ** (torch.arange(0, d, 2, device="cuda").float() / d), 4 * page)
    table = torch.randperm(size, generator=gen, device="cuda").to(torch.int32).view(size, 1)
    out = []
    for rows in (m, size):
        positions = (torch.arange(rows, device="cuda") % page).to(torch.int32)
        pages = [torch.zeros(shape(size, nkv, page, d), dtype=torch.bfloat16, device="cuda") for shape in (ops.key_pages_shape, ops.value_pages_shape)]
        q = lin.rope_append(x[:rows], ops.RopeAppend(positions, torch.arange(rows, device="cuda", dtype=torch.int32), table, cos, sin, *pages, nq, nkv, d, page))
        out.append((q, *(p[table[:m, 0].long()] for p in pages)))
    assert torch.equal(out[0][0], out[1][0][:m])
    assert torch.equal(out[0][1], out[1][1]) and torch.equal(out[0][2], out[1][2])


def test_product_and_pass_in_one_call():
    """The bits of the two calls, and what they refuse is refused."""
    x, w, gen = _case(33, 256, 192, 5)
    residual, weight = torch.randn((33, 256), generator=gen, device="cuda").bfloat16(), torch.randn((256,), generator=gen, device="cuda")
    for got, want in zip(ops.split_linear_add_rmsnorm(x, w, residual, weight, 1e-5), ops.split_add_rmsnorm(ops.gemm_split(x, w), residual, weight, 1e-5)):
        assert torch.equal(got, want)
    positions, table = torch.arange(33, device="cuda", dtype=torch.int32), torch.randperm(3, generator=gen, device="cuda").to(torch.int32).view(1, 3)
    cos, sin = ops.rope_table(1.0 / 10000 ** (torch.arange(0, 32, 2, device="cuda").float() / 32), 48)
    pages = [[torch.zeros(shape(3, 2, 16, 32), dtype=torch.bfloat16, device="cuda") for shape in (ops.key_pages_shape, ops.value_pages_shape)] for _ in range(2)]
    rope = [ops.RopeAppend(positions, torch.zeros_like(positions), table, cos, sin, *p, 4, 2, 32, 16) for p in pages]
    assert torch.equal(ops.split_linear_rope_append(x, w, rope[0]), ops.split_rope_append(ops.gemm_split(x, w), rope[1]))
    assert torch.equal(pages[0][0], pages[1][0]) and torch.equal(pages[0][1], pages[1][1])
    for bad in ((x[:, :96], w[:, :96].contiguous(), residual, weight), (x, w[:60], residual, weight), (x, w, residual[:30], weight),
                (x, w, residual, weight[:100]), (x, w, residual.float(), weight), (x[:, 1:65], w[:, :64].contiguous(), residual, weight)):
        with pytest.raises(ops.KernelError):
            ops.split_linear_add_rmsnorm(*bad, 1e-5)
    rope[0].positions = positions[:30]
    with pytest.raises(ops.KernelError):
        ops.split_linear_rope_append(x, w, rope[0])


def test_what_is_refused():
    x, w, _ = _case(4, 64, 128, 1)
    for bad in ((x[:, :96], w[:, :96].contiguous()), (x, w[:60]), (torch.cat([x] * 65), w), (x.float(), w.float()), (x[:, 1:65], w[:, :64].contiguous())):
        with pytest.raises(ops.KernelError):
            ops.gemm_split(*bad)
