"""Heads of one size, all of each rotated, normed and appended 16 bytes at a time, against the kernel that takes any heads (which rows that
start at no multiple of 16 bytes go to): sizes at which a lane has its most pieces and one more, tokens that fill no workgroup, both pairs."""

import pytest
import torch

from tokasaurus_amd.kernels import ops

pytestmark = pytest.mark.gpu


# pieces of 8 elements a token: 4, 18, 256 (four a lane), 264, 512, 768, 1,024 (the most), 1,026 (the general kernel's)
@pytest.mark.parametrize("nq,nkv,d", [(2, 0, 16), (5, 2, 16), (16, 8, 64), (9, 4, 128), (33, 0, 64), (16, 8, 128), (32, 8, 128), (64, 32, 64), (40, 12, 128), (1, 1, 32), (171, 171, 16)])
@pytest.mark.parametrize("norm", ["none", "head", "row", "queries", "keys"])
@pytest.mark.parametrize("halves", [False, True])
@pytest.mark.parametrize("n", [5, 515])
def test_wide_pieces_follow_the_general_kernel(nq, nkv, d, norm, halves, n):
    P, g = 8, torch.Generator(device="cuda").manual_seed(nq + d + n)
    write, rand = nkv > 0, lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    pages, per_head = -(-n // P) + 2, norm in ("head", "queries")
    width = (nq + 2 * nkv) * d
    rows = rand(n, width).bfloat16()
    weight = lambda heads: 1 + 0.2 * rand(d if per_head else heads * d)  # noqa: E731
    qw = weight(nq) if norm in ("head", "row", "queries") else None
    kw = weight(nkv) if write and norm in ("head", "row", "keys") else None
    freq = 10000.0 ** (-torch.arange(0, d, 2, device="cuda").float() / d)
    split = n // 3  # two requests
    req = torch.tensor([0] * split + [1] * (n - split), dtype=torch.int32, device="cuda")
    pos = torch.cat([torch.arange(split), torch.arange(n - split)]).int().cuda()
    table = torch.randperm(2 * pages, generator=torch.Generator().manual_seed(n)).int().cuda().view(2, pages)
    results = []
    for stride in (width, width + 4):
        x = torch.zeros((n, stride), dtype=torch.bfloat16, device="cuda")
        x[:, :width] = rows
        kc = torch.zeros(ops.key_pages_shape(2 * pages, max(nkv, 1), P, d), dtype=torch.bfloat16, device="cuda")
        vc = torch.zeros(ops.value_pages_shape(2 * pages, max(nkv, 1), P, d), dtype=torch.bfloat16, device="cuda")
        ops.qk_prepare(x[:, :width], pos, req, table, qw, kw, 1e-6, freq, kc if write else None, vc if write else None, nq, max(nkv, 1) if not write else nkv,
                       d, d, P, write_cache=write, per_head=per_head, pair_halves=halves, rotation_scale=1.25)
        results.append((x[:, : nq * d], kc, vc))
    (q, k, v), (want_q, want_k, want_v) = results
    assert torch.equal(v, want_v)
    for got, want in ((q, want_q), (k, want_k)):
        if norm == "none":  # the same operations
            assert torch.equal(got, want)
            continue
        # the squares' sum in another order: a 32-bit factor that differs in its last places, which may turn a rounding to bfloat16 (one of its
        # units, 2^-7 of the smaller number) and where a rotation cancels is seen against its operands, of up to six
        got, want = got.double(), want.double()
        assert bool(((got - want).abs() <= 2.0 ** -7 * want.abs() + 6 * 1.25 * 2.0 ** -20).all())
