"""The weight-streaming and the streamed gate and up products with a norm in front, at the edges of what is asked for early: rows
beyond a wavefront's first, partial sums that are as many as the lanes take, more, and no multiple of 4; a rotation
behind a folded K; and the norm by itself where the pieces of a row that a thread holds change in number."""

from __future__ import annotations

import pytest
import torch

from tokasaurus_amd.kernels import ops

pytestmark = pytest.mark.gpu


def _norm(m, k, parts, gen):
    x = torch.randn((m, k), generator=gen, device="cuda").bfloat16()
    sumsq = torch.rand((m, parts), generator=gen, device="cuda") * 2 * k / parts
    return ops.Prenorm(x, sumsq), x.double() / torch.sqrt(sumsq.double().sum(1, keepdim=True) / k + 1e-5)


@pytest.mark.parametrize("m", [1, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("parts", [4, 252, 256, 260, 6])
def test_norm_in_front(m, parts):
    """32-bit sums of k products and of the partial sums, the factor's root and division: (k + parts + 8) 2^-24 of the sum of the
    magnitudes; the activation behind gate and up rounds three times to 8 bits."""
    gen = torch.Generator(device="cuda").manual_seed(m + parts)
    n, k = 264, 448
    pre, rows = _norm(m, k, parts, gen)
    w = (torch.randn((2 * n, k), generator=gen, device="cuda") / k ** 0.5).bfloat16()
    want, size = rows @ w.double().T, rows.abs() @ w.double().abs().T
    for kw in ({}, {"tile_rows": 8}, {"staged": 1}):
        got = ops.gemm_skinny_bf16(pre.scaled, w, prenorm=pre, norm_eps=1e-5, out_f32=True, **kw)
        assert ((got.double() - want).abs() <= (k + parts + 8) * 2.0 ** -24 * size).all(), kw
    got = ops.gemm_skinny_bf16(pre.scaled, w, prenorm=pre, norm_eps=1e-5, swiglu=True, staged=2)
    gate, up = want[:, :n], want[:, n:]
    # a rounding to 8 significant bits is off by 2^-8 of the value at most: gate (silu's slope is at most 1.1), up, silu, the product
    s = torch.nn.functional.silu(gate)
    bound = 2.0 ** -8 * (1.1 * gate.abs() * up.abs() + 3 * (s * up).abs()) * 1.1 + 1e-6
    assert ((got.double() - s * up).abs() <= bound).all()


@pytest.mark.parametrize("weight_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n", [1, 3, 9, 200, 201])
@pytest.mark.parametrize("begin", [0, 1, 2])
def test_weights_of_the_norm_behind_that_begin_and_end_anywhere(weight_dtype, n, begin):
    """Weights that start 0, 1 and 2 elements behind a multiple of 16 bytes and are no whole words: the emitted rows are x w, rounded once,
    and the partial sums those of the rounded rows (16 squares of one sign: 16 roundings of 2^-24)."""
    gen = torch.Generator(device="cuda").manual_seed(n + begin)
    m, k = 3, 96
    a, w, res = (torch.randn(s, generator=gen, device="cuda").bfloat16() for s in ((m, k), (n, k), (m, n)))
    weight = (1 + torch.randn((n + begin,), generator=gen, device="cuda")).to(weight_dtype)[begin:]
    x, pre = ops.gemm_skinny_bf16(a, w, residual=res, emit_weight=weight)
    assert torch.equal(pre.scaled, (weight.float() * x.float()).bfloat16())
    assert torch.allclose(pre.sumsq.sum(1), x.float().pow(2).sum(1), rtol=16 * 2.0 ** -24 + n * 2.0 ** -24, atol=0)


@pytest.mark.parametrize("m", [1, 2])
def test_tiles_of_8_for_one_and_two_rows_where_they_are_folded(m):
    """4,096 outputs fill the compute units with tiles of 16 as well: an inner size of no multiple of 64, two tiles a wavefront, and a product that
    is asked not to fold K take those; and the partial sums are as many as the caller is told."""
    from tokasaurus_amd.kernels.library import load

    parts = load("mfma").tk_gemm_skinny_parts
    assert parts(m, 4096, 2048, 0, 0, 1) == 512
    assert parts(m, 4096, 2080, 0, 0, 1) == parts(m, 4096, 2048, 2, 0, 1) == parts(m, 4096, 2048, 0, 0, 0) == 256
    gen = torch.Generator(device="cuda").manual_seed(m)
    for k in (64, 96):
        a, w, res, weight = (torch.randn(s, generator=gen, device="cuda").bfloat16() for s in ((m, k), (4096, k), (m, 4096), (4096,)))
        for kw in ({}, {"tiles": 2}, {"fold": False}):
            x, pre = ops.gemm_skinny_bf16(a, w, residual=res, emit_weight=weight, **kw)
            want = (a.double() @ w.double().T).bfloat16().double() + res.double()
            assert ((x.double() - want).abs() <= 2.0 ** -7 * (want.abs() + (a.double().abs() @ w.double().abs().T))).all()
            assert torch.equal(pre.scaled, (weight.float() * x.float()).bfloat16())
            assert torch.allclose(pre.sumsq.sum(1), x.float().pow(2).sum(1), rtol=4096 * 2.0 ** -24, atol=0)


@pytest.mark.parametrize("m", [1, 9, 17, 40])
@pytest.mark.parametrize("steps", [1, 2, 3, 5, 7, 8, 9, 10, 15, 16, 17])
def test_steps_that_are_left_behind_whole_groups(m, steps):
    """Walks of one wavefront, and of two of uneven length, over fewer steps than a group of loads, whole groups and some more: sums of k products
    in 32-bit, k 2^-24 of the sum of the magnitudes; behind gate and up three roundings to 8 bits more."""
    gen = torch.Generator(device="cuda").manual_seed(m + steps)
    k, n = 32 * steps, 72
    pre, rows = _norm(m, k, 8, gen)
    w = torch.randn((2 * n, k), generator=gen, device="cuda").bfloat16()
    want, size = rows @ w.double().T, rows.abs() @ w.double().abs().T
    for waves in (1, 2):
        got = ops.gemm_skinny_bf16(pre.scaled, w, out_f32=True, waves_k=waves, fold=steps % 2 == 0)
        plain, plain_size = pre.scaled.double() @ w.double().T, pre.scaled.double().abs() @ w.double().abs().T
        assert ((got.double() - plain).abs() <= (k + 8) * 2.0 ** -24 * plain_size).all()
        got = ops.gemm_skinny_bf16(pre.scaled, w, prenorm=pre, norm_eps=1e-5, out_f32=True, waves_k=waves)
        assert ((got.double() - want).abs() <= (k + 16) * 2.0 ** -24 * size).all()
        got = ops.gemm_skinny_bf16(pre.scaled, w, prenorm=pre, norm_eps=1e-5, swiglu=True, staged=0, waves_k=waves)
        gate, up, slack = want[:, :n], want[:, n:], (k + 16) * 2.0 ** -24
        s = torch.nn.functional.silu(gate)
        bound = 2.0 ** -8 * (1.1 * gate.abs() * up.abs() + 3 * (s * up).abs()) * 1.1 + 2 * slack * (size[:, :n] * up.abs() + s.abs() * size[:, n:]) + 1e-6
        assert ((got.double() - s * up).abs() <= bound).all()


@pytest.mark.parametrize("begin", [1, 2, 3])
def test_rows_for_the_norm_behind_that_begin_anywhere(begin, monkeypatch):
    """Memory for x w that starts 2, 4 and 6 bytes behind a multiple of 8: the same values."""
    gen = torch.Generator(device="cuda").manual_seed(begin)
    a, w, res, weight = (torch.randn(s, generator=gen, device="cuda").bfloat16() for s in ((3, 96), (200, 96), (3, 200), (200,)))
    want = ops.gemm_skinny_bf16(a, w, residual=res, emit_weight=weight)
    made = ops.Prenorm
    monkeypatch.setattr(ops, "Prenorm", lambda scaled, sumsq: made(torch.empty((603,), dtype=scaled.dtype, device="cuda")[begin:][:600].view(3, 200), sumsq))
    got = ops.gemm_skinny_bf16(a, w, residual=res, emit_weight=weight)
    assert got[1].scaled.data_ptr() % 8 == 2 * begin
    assert torch.equal(got[0], want[0]) and torch.equal(got[1].scaled, want[1].scaled) and torch.equal(got[1].sumsq, want[1].sumsq)


@pytest.mark.parametrize("m", [1, 3, 8, 9])
@pytest.mark.parametrize("k", [64, 448, 576, 2048])
def test_rotation_behind_a_folded_inner_size(m, k):
    """Queries and pages as the plain product and the rotation kernel leave them, up to the order of the product's 32-bit sums: a rounding
    of 8 bits falls the other way at most, which is 2^-8 of a pair's length."""
    gen = torch.Generator(device="cuda").manual_seed(m + k)
    nq, nkv, d, page = 4, 2, 48, 16
    width = (nq + 2 * nkv) * d
    pre, rows = _norm(m, k, 64, gen)
    w = (torch.randn((width, k), generator=gen, device="cuda") / k ** 0.5).bfloat16()
    positions = torch.randint(0, 90, (m,), generator=gen, device="cuda").to(torch.int32)
    req = torch.arange(m, device="cuda", dtype=torch.int32)
    table = torch.randperm(m * 6, generator=gen, device="cuda").to(torch.int32).view(m, 6)
    cos, sin = ops.rope_table(1.0 / 10000 ** (torch.arange(0, d, 2, device="cuda").float() / d), 96)
    pages = [(torch.zeros(ops.key_pages_shape(6 * m, nkv, page, d), device="cuda", dtype=torch.bfloat16),
              torch.zeros(ops.value_pages_shape(6 * m, nkv, page, d), device="cuda", dtype=torch.bfloat16)) for _ in range(2)]
    ropes = [ops.RopeAppend(positions, req, table, cos, sin, *p, nq, nkv, d, page) for p in pages]
    stacked = (rows @ w.double().T).bfloat16()
    ops.rope_append(stacked, positions, req, table, cos, sin, *pages[0], nq, nkv, d, page)
    q = ops.gemm_skinny_bf16(pre.scaled, w, rope=ropes[1], tile_rows=8, prenorm=pre, norm_eps=1e-5)
    largest = float(stacked.double().abs().max())
    for got, want in ((q, stacked[:, : nq * d]), (pages[1][0], pages[0][0]), (pages[1][1], pages[0][1])):
        assert float((got.double() - want.double()).abs().max()) <= 2.0 ** -7 * largest


@pytest.mark.parametrize("d,split,waves", [(64, 128, 4), (64, 96, 3), (64, 2048, 16), (128, 256, 4), (128, 160, 5), (128, 4096, 8)])
@pytest.mark.parametrize("window", [0, 70])
def test_wavefronts_share_the_keys_that_a_split_has(d, split, waves, window):
    """Requests that end anywhere in a split (or whose window begins there), against 64-bit attention: keys, values and weights have 8
    significant bits, and the sums are 32-bit: 2^-7 of the weighted magnitudes."""
    nq, nkv, page = 8, 2, 16
    lens = [1, 31, 32, 33, 95, 127, 128, 129, 200, 400]
    gen = torch.Generator(device="cuda").manual_seed(d + split)
    rand = lambda *s: torch.randn(s, generator=gen, device="cuda").bfloat16()  # noqa: E731
    pages = [-(-n // page) for n in lens]
    kc, vc = rand(*ops.key_pages_shape(sum(pages), nkv, page, d)), rand(*ops.value_pages_shape(sum(pages), nkv, page, d))
    table, at = torch.zeros((len(lens), 32), dtype=torch.int32), 0
    for i, n in enumerate(pages):
        table[i, :n] = torch.arange(at, at + n)
        at += n
    q = rand(len(lens), nq * d)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    got = ops.paged_attention_mfma(q, kc, vc, table.cuda(), i32(range(len(lens) + 1)), i32(lens), i32(range(len(lens))), i32([0] * len(lens)), 1,
                                   nq, nkv, d, page, 512, split, waves=waves, window=window)
    for i, n in enumerate(lens):
        mine = table[i, : pages[i]].long().cuda()
        k = kc[mine].double().permute(1, 0, 3, 2, 4).reshape(nkv, -1, d)[:, max(0, n - window) if window else 0 : n]
        v = vc[mine].double().permute(1, 0, 2, 4, 3).reshape(nkv, -1, d)[:, max(0, n - window) if window else 0 : n]
        k, v = k.repeat_interleave(nq // nkv, 0), v.repeat_interleave(nq // nkv, 0)
        p = torch.softmax((k @ q[i].double().view(nq, d, 1))[..., 0] * d ** -0.5, -1)
        want, size = (p[:, None] @ v)[:, 0], (p[:, None] @ v.abs())[:, 0]
        assert ((got[i].double().view(nq, d) - want).abs() <= 2.0 ** -7 * size + 1e-6).all(), n


@pytest.mark.parametrize("d,split,waves", [(64, 128, 4), (64, 96, 3), (64, 4096, 8), (128, 256, 4), (128, 160, 5), (128, 4096, 8)])
@pytest.mark.parametrize("window", [0, 70])
def test_wavefronts_share_the_keys_that_are_there(d, split, waves, window, monkeypatch):
    """The same where a request's keys, not the split, are shared evenly."""
    attention = ops.paged_attention_mfma
    monkeypatch.setattr(ops, "paged_attention_mfma", lambda *a, **kw: attention(*a, **kw, even=True))
    test_wavefronts_share_the_keys_that_a_split_has(d, split, waves, window)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("pieces", [1, 255, 256, 257, 511, 512, 513, 1024, 1025])
def test_rows_held_in_registers_by_the_norm(dtype, pieces):
    """Where a thread's pieces of 16 bytes go from one to two to four and to a loop, and where its last one lies behind the row's end."""
    hidden = pieces * 16 // dtype.itemsize
    gen = torch.Generator().manual_seed(pieces)
    x, r = (torch.randn((3, hidden), generator=gen).to(dtype) for _ in range(2))
    for weight_dtype in {dtype, torch.float32}:
        w = (1 + 0.1 * torch.randn((hidden,), generator=gen)).to(weight_dtype)
        stream, normed = (t.cpu() for t in ops.add_rmsnorm(x.cuda(), r.cuda(), w.cuda(), 1e-5))
        assert torch.equal(stream, x + r)
        rows = stream.double()
        want = w.double() * rows / torch.sqrt(rows.pow(2).mean(1, keepdim=True) + 1e-5)
        # a row's sum of squares is good to (hidden / 256 + 16) roundings; the normed value and its product with the weight are rounded (half an eps each)
        limit = want.abs() * (1.02 * torch.finfo(dtype).eps + (hidden / 256 + 24) * 2.0 ** -23)
        assert ((normed.double() - want).abs() <= limit).all()
        assert torch.equal(ops.rmsnorm(stream.cuda(), w.cuda(), 1e-5).cpu(), normed)
