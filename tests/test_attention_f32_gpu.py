"""32-bit grouped-query attention takes the matrix-core kernel where its sizes allow: against the plain kernel, over steps of
portions, of single tokens and of both, windows, groups, head and page sizes, with NaN in every place of the pages that holds
no token of the step's requests."""

import pytest
import torch

from test_parts_gpu import context
from tokasaurus_amd.kernels import ops
from tokasaurus_amd.parts import MIXERS, CacheView, PartSpec
from tokasaurus_amd.parts.linear import Placer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads", [(4, 4, 16), (6, 2, 64), (8, 1, 32), (8, 2, 128),  # groups of 1, 3, 8 and 4
                                   (9, 3, 112), (4, 2, 48), (8, 2, 80), (4, 4, 96), (4, 1, 144)])  # heads that fill no power of two of blocks
@pytest.mark.parametrize("page,window", [(16, 0), (32, 21), (64, 300)])
@pytest.mark.parametrize("step", [([40, 17], [0, 9]), ([1, 1, 1], [0, 15, 700]), ([33, 2, 1, 1], [0, 290, 31, 512])])
def test_matches_the_plain_kernel(heads, page, window, step, monkeypatch):
    nq, nkv, d = heads
    q_lens, starts = step
    g = torch.Generator().manual_seed(sum(q_lens) + d)
    H = 64
    rand = lambda *s: torch.randn(s, generator=g)  # noqa: E731
    tensors = {"q.w": rand(nq * d, H) * 0.2, "k.w": rand(nkv * d, H) * 0.2, "v.w": rand(nkv * d, H) * 0.2, "o.w": rand(H, nq * d) * 0.1}
    mixer = MIXERS.build(PartSpec("paged_attention", {
        "hidden_size": H, "num_heads": nq, "num_kv_heads": nkv, "head_dim": d, "window": window,
        "names": {"q": "q.w", "k": "k.w", "v": "v.w", "o": "o.w"}}))
    mixer.load(tensors, Placer(torch.float32, torch.device("cuda")))
    blocks = [-(-(s + n) // page) for s, n in zip(starts, q_lens)]
    tables, at = [], 0
    for b in blocks:
        tables.append(list(range(at, at + b)))
        at += b
    keys = torch.full(ops.key_pages_shape(at + 1, nkv, page, d), float("nan"), device="cuda")
    values = torch.full(ops.value_pages_shape(at + 1, nkv, page, d), float("nan"), device="cuda")
    fill = [torch.randn((s, H), generator=g) for s in starts]
    if any(starts):  # the past, as one step of portions
        held = [i for i, s in enumerate(starts) if s]
        ctx, table = context([starts[i] for i in held], [0] * len(held), [tables[i] for i in held], torch.float32)
        order = sorted(range(len(held)), key=lambda i: starts[held[i]] == 1)  # (a step's single tokens come last)
        x = torch.cat([fill[held[i]] for i in order]).cuda()
        mixer.forward(x, x, ctx, CacheView(keys, values, table, page), None, None)
    x = torch.randn((sum(q_lens), H), generator=g).cuda()
    got = []
    for takes in (True, False):
        ctx, table = context(q_lens, starts, tables, torch.float32)
        if not takes:
            monkeypatch.setattr(ops, "attention_tile_f32_fits", lambda *a: False)
        else:
            assert ops.attention_tile_f32_fits(nq, nkv, d, d, page)
        out = mixer.forward(x, torch.zeros_like(x), ctx, CacheView(keys, values, table, page), None, None)
        got.append((out[0] if isinstance(out, tuple) else out).double())
    # both sum at most 1,032 keys and 1,024 outputs in 32-bit, in other orders: (1032 + 1024) 2^-24 of the terms' magnitude,
    # which for these sizes is below four times the outputs' own root mean square
    assert torch.isfinite(got[0]).all()
    assert float((got[0] - got[1]).abs().max()) <= 2056 * 2.0 ** -24 * 4 * float(got[1].pow(2).mean().sqrt())
