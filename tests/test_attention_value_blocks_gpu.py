"""Paged attention in 32-bit arithmetic for value heads of every number of 16-element blocks, with key heads on both sides of
the kernel's sizes: in both storage types, with a tile a wavefront, tiles shared by a workgroup's wavefronts, and keys cut
among workgroups.  Against sums in 64-bit."""

from __future__ import annotations

import pytest
import torch

from tokasaurus_amd.kernels import ops

pytestmark = pytest.mark.gpu

LENS, PORTIONS, PAGE, NQ, NKV = [45, 300], [45, 20], 32, 4, 2


def _paged(dk, dv, dtype, gen):
    """Keys and values in pages in shuffled order; every place behind a request's end is NaN."""
    pages = [-(-n // PAGE) for n in LENS]
    order = (torch.randperm(sum(pages), generator=gen) + 1).tolist()
    table = torch.zeros((len(LENS), max(pages)), dtype=torch.int32)
    kc = torch.full(ops.key_pages_shape(sum(pages) + 1, NKV, PAGE, dk), float("nan"), dtype=dtype)
    vc = torch.full(ops.value_pages_shape(sum(pages) + 1, NKV, PAGE, dv), float("nan"), dtype=dtype)
    keys = [torch.randn((n, NKV, dk), generator=gen).to(dtype) for n in LENS]
    values = [torch.randn((n, NKV, dv), generator=gen).to(dtype) for n in LENS]
    for r, n in enumerate(LENS):
        for i in range(pages[r]):
            p = table[r, i] = order.pop()
            m = min(PAGE, n - i * PAGE)
            k = torch.full((PAGE, NKV, dk), float("nan"), dtype=dtype)
            v = torch.full((PAGE, NKV, dv), float("nan"), dtype=dtype)
            k[:m], v[:m] = keys[r][i * PAGE: i * PAGE + m], values[r][i * PAGE: i * PAGE + m]
            kc[p] = k.view(PAGE, NKV, dk // 8, 8).permute(1, 2, 0, 3)
            vc[p] = v.view(PAGE // 4, 4, NKV, dv).permute(2, 0, 3, 1)
    return keys, values, kc, vc, table


@pytest.mark.parametrize("form", [{"split": False}, {"split": True}, {"split": True, "key_chunk": 128, "longest": max(LENS)}],
                         ids=["tile a wavefront", "shared tiles", "keys cut"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["float32", "bfloat16"])
@pytest.mark.parametrize("dk,dv", [(16, 16), (32, 32), (40, 48), (72, 48), (200, 48), (64, 64), (80, 80), (64, 96), (96, 96), (24, 112), (64, 112),
                                   (112, 112), (192, 112), (128, 128), (144, 144), (64, 176), (192, 192), (240, 240), (64, 240), (256, 256)])
def test_every_number_of_value_blocks(dk, dv, dtype, form):
    gen = torch.Generator().manual_seed(dk * 1000 + dv)
    keys, values, kc, vc, table = _paged(dk, dv, dtype, gen)
    q = torch.randn((sum(PORTIONS), NQ, dk), generator=gen).to(dtype)
    start = [0, PORTIONS[0], sum(PORTIONS)]
    tiles = [(r, a) for r in range(2) for a in range(start[r], start[r + 1], 16)]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    scale = dk ** -0.5
    out = ops.attention_tile_f32(q.cuda().view(-1, NQ * dk), kc.cuda(), vc.cuda(), table.cuda(), i32(start), i32(LENS),
                                 i32([r for r, _ in tiles]), i32([a for _, a in tiles]), NQ, NKV, dk, dv, PAGE, 1, scale=scale, **form)
    out = out.cpu().double().view(-1, NQ, dv)
    for r, n in enumerate(LENS):
        Q = q[start[r]: start[r + 1]].double().permute(1, 0, 2)
        K = keys[r].double().repeat_interleave(NQ // NKV, 1).permute(1, 0, 2)
        V = values[r].double().repeat_interleave(NQ // NKV, 1).permute(1, 0, 2)
        s = Q @ K.transpose(1, 2) * float(torch.tensor(scale, dtype=torch.float32))
        seen = torch.arange(n)[None] <= torch.arange(n - PORTIONS[r], n)[:, None]
        w = torch.softmax(s.masked_fill(~seen, float("-inf")), -1)
        want, size = (w @ V).permute(1, 0, 2), (w @ V.abs()).permute(1, 0, 2)
        # scores are 32-bit sums of dk products (their error moves a weight by as much, relatively), the sums over the keys
        # 32-bit sums of n; a bfloat16 result is rounded once more (up to 2^-8 of it)
        reach = float((Q.abs() @ K.abs().transpose(1, 2)).max()) * scale
        limit = size * (n + 64 + dk * reach) * 2.0 ** -23 + (want.abs() * 2.0 ** -8 if dtype == torch.bfloat16 else 0)
        worst = ((out[start[r]: start[r + 1]] - want).abs() - limit).amax((0, 1))
        assert float(worst.max()) <= 0, f"request {r}: element {int(worst.argmax())} of {dv}"


@pytest.mark.parametrize("form", [{"split": False}, {"split": True}, {"split": True, "key_chunk": 128, "longest": max(LENS)}],
                         ids=["tile a wavefront", "shared tiles", "keys cut"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["float32", "bfloat16"])
@pytest.mark.parametrize("mask", [{}, {"window": 21}, {"section": 25}], ids=["all", "window", "sections"])
def test_what_is_not_finite_stays_with_those_who_see_it(mask, dtype, form):
    """An infinite value, a NaN among the values and keys that are all NaN reach the tokens that see them and no others of their
    tile, as in the plain kernel."""
    gen = torch.Generator().manual_seed(3)
    d = 64
    _, _, kc, vc, table = _paged(d, d, dtype, gen)
    for r, at, x in ((0, 37, float("inf")), (1, 285, float("nan"))):
        vc[table[r, at // PAGE], :, at % PAGE // 4, 5, at % 4] = x
    for at in range(16):
        kc[table[0, 0], 1, :, at] = float("nan")
    q = torch.randn((sum(PORTIONS), NQ * d), generator=gen).to(dtype).cuda()
    start = [0, PORTIONS[0], sum(PORTIONS)]
    tiles = [(r, a) for r in range(2) for a in range(start[r], start[r + 1], 16)]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    req = i32([r for r in range(2) for _ in range(PORTIONS[r])])
    pos = i32([p for r in range(2) for p in range(LENS[r] - PORTIONS[r], LENS[r])])
    kc, vc, table = kc.cuda(), vc.cuda(), table.cuda()
    want = ops.paged_attention_generic(q, kc, vc, table, req, pos, NQ, NKV, d, PAGE, scale=0.125, **mask)
    got = ops.attention_tile_f32(q, kc, vc, table, i32(start), i32(LENS), i32([r for r, _ in tiles]), i32([a for _, a in tiles]),
                                 NQ, NKV, d, d, PAGE, 1, scale=0.125, **mask, **form)
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
    assert bool(torch.isinf(want).any()) and bool(torch.isnan(want).any())
    held = torch.isfinite(want)
    # each kernel within the bound of the test above, with a result's size below the largest value's
    reach = float((q.float().abs().view(-1, NQ, d).sum(-1).max() * kc.float().nan_to_num(0).abs().max())) * 0.125
    largest = float(vc.float().nan_to_num(0, 0, 0).abs().max())
    limit = 2 * largest * (max(LENS) + 64 + d * reach) * 2.0 ** -23 + (largest * 2.0 ** -8 if dtype == torch.bfloat16 else 0)
    assert float((got[held].double() - want[held].double()).abs().max()) <= limit
