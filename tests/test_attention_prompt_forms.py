"""Prompt portions whose keys the wavefronts of a workgroup share: single and neighbouring tiles against pairs in a wavefront, and when they are taken."""

import pytest
import torch

from tokasaurus_amd.kernels import ops


def test_which_form_prompt_portions_take():
    form = ops.attention_prompt_form
    assert form(608, 64, 5000) == form(448, 128, 100) == (1, 2)
    assert form(609, 64, 699) == form(449, 128, 699) == (2, 1) and form(609, 64, 700) == form(3072, 128, 700) == (2, 2)
    assert form(3073, 64, 4000) == (2, 1)


@pytest.mark.parametrize("q_lens,kv_lens,unit,form", [([1024, 1000, 1300], [1024, 1200, 1300], 4, 2), ([90, 33, 60], [90, 500, 64], 1, 1), ([700, 720], [700, 720], 1, 2)])
def test_longest_walks_start_first(monkeypatch, q_lens, kv_lens, unit, form):
    """The plan's tiles are those of every portion, each once, in the order of the keys they reach."""
    from types import SimpleNamespace

    from tokasaurus_amd.parts import attention

    monkeypatch.setattr(attention, "upload", lambda values, dtype, device: torch.tensor(values, dtype=dtype))
    start = [sum(q_lens[:i]) for i in range(len(q_lens) + 1)]
    ctx = SimpleNamespace(extras={}, num_requests=len(q_lens), host_q_start=start, host_kv_len=kv_lens, max_kv_len=max(kv_lens), device=torch.device("cpu"))
    (launch,) = attention.attention_plan(ctx, 4, 8, 64, 16).launches
    req, row0 = launch.tile_req.tolist(), launch.tile_row0.tolist()
    assert launch.row_tiles == form and (launch.grouped > 0) == (unit == 4)
    fill = ops.ATTENTION_GROUP if unit == 4 else 1
    want = ops.attention_tiles(q_lens, 4, form, fill=fill)
    assert sorted(zip(req, row0)) == sorted(zip(want[0], want[1]))
    reach = [max(kv_lens[req[j]] - q_lens[req[j]] + row0[j] // 4 for j in range(i, i + unit)) for i in range(0, len(req), unit)]
    assert reach == sorted(reach, reverse=True)
    assert all(len(set(req[i : i + unit])) == 1 for i in range(0, len(req), unit))


# portions whole, one token over a step, after a past; windows that end a walk inside a step; pages of fewer keys than a block has; every
# wavefront with keys, and wavefronts without
@pytest.mark.gpu
@pytest.mark.parametrize("lens,portions,nq,nkv,d,page,window", [([97, 400], [97, 400], 8, 2, 64, 16, 0), ([33, 1, 640], [33, 1, 33], 4, 4, 128, 16, 0),
                                                                ([300], [300], 6, 2, 112, 4, 0), ([500], [400], 4, 1, 16, 8, 70), ([900], [450], 3, 1, 128, 32, 333)])
def test_shared_keys_give_the_same_as_pairs(lens, portions, nq, nkv, d, page, window):
    g = torch.Generator(device="cuda").manual_seed(sum(lens) + d)
    pages = -(-max(lens) // page)
    rand = lambda shape: torch.randn(shape, generator=g, device="cuda").bfloat16()  # noqa: E731
    keys, values = rand(ops.key_pages_shape(pages * len(lens), nkv, page, d)), rand(ops.value_pages_shape(pages * len(lens), nkv, page, d))
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    table = torch.randperm(pages * len(lens), generator=torch.Generator().manual_seed(d)).int().cuda().view(len(lens), pages)
    start = [sum(portions[:i]) for i in range(len(lens) + 1)]
    q, bound = rand((start[-1], nq * d)), -(-max(lens) // 256) * 256

    def run(row_tiles, waves, pair):
        req, row0, row1 = ops.attention_tiles(portions, nq // nkv, row_tiles, pair=pair)
        if not pair:
            req, row0 = req[::-1], row0[::-1]
        return ops.paged_attention_mfma(q, keys, values, table, i32(start), i32(lens), i32(req), i32(row0), row_tiles, nq, nkv, d, page, max(lens), bound,
                                        window=window, waves=waves, tile_row1=None if row1 is None else i32(row1), even=waves > 1).double()

    want = run(2, 1, True)
    for row_tiles, waves in ((1, 2), (2, 2), (2, 4), (1, 8)):
        # the weights of a softmax's terms rounded to bfloat16 under another maximum (2^-8 of each, values of up to five, in root mean square a
        # tenth of that), and the result's own rounding
        got = run(row_tiles, waves, False)
        assert bool(((got - want).abs() <= 2.0 ** -7 * want.abs() + 5 * 2.0 ** -8).all()), (row_tiles, waves)
        assert float((got - want).norm() / want.norm()) <= 2.0 ** -7, (row_tiles, waves)


FORMS = {"pairs": (2, 1, 0), "single": (1, 2, 0), "neighbours": (2, 2, 0), "group": (2, 1, 1), "sets": (2, 1, 2), "decode": (1, 2, 0)}


def of_products(rows, form):
    """One request of n keys, of which key i has the product rows[i] / log2(e) with every query: what the kernel gives for all its
    tokens (``decode``: for the last), and what a softmax in 64 bits does."""
    nq, nkv, d, page, n = 4, 2, 64, 16, rows.numel()
    g = torch.Generator(device="cuda").manual_seed(3)
    pages = -(-n // page)
    k = torch.zeros((n, nkv, d), device="cuda")
    k[:, :, 0] = (rows / 1.4427).bfloat16().float()[:, None]  # (two pieces of a bfloat16 number each: what is left of the first, by another element)
    k[:, :, 1] = (rows / 1.4427 - k[:, 0, 0]).bfloat16().float()[:, None]
    q = torch.zeros((n, nq, d), device="cuda")
    q[..., 0] = q[..., 1] = 1
    v = torch.randn((n, nkv, d), generator=g, device="cuda").bfloat16()
    keys = torch.zeros(ops.key_pages_shape(pages, nkv, page, d), dtype=torch.bfloat16, device="cuda")
    values = torch.zeros(ops.value_pages_shape(pages, nkv, page, d), dtype=torch.bfloat16, device="cuda")
    pad = pages * page - n
    kp, vp = (torch.nn.functional.pad(x, (0, 0, 0, 0, 0, pad)).view(pages, page, nkv, d) for x in (k.bfloat16(), v))
    keys.view(pages, nkv, d // 8, page, 8).copy_(kp.view(pages, page, nkv, d // 8, 8).permute(0, 2, 3, 1, 4))
    values.view(pages, nkv, page // 4, d, 4).copy_(vp.view(pages, page // 4, 4, nkv, d).permute(0, 3, 1, 4, 2))
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    row_tiles, waves, grouped = FORMS[form]
    tokens = 1 if form == "decode" else n
    req, row0, row1 = ops.attention_tiles([tokens], nq // nkv, row_tiles, pair=form == "pairs", fill=ops.ATTENTION_GROUP if grouped else 1)
    out = ops.paged_attention_mfma(q[-tokens:].reshape(tokens, -1).bfloat16(), keys, values, torch.arange(pages, device="cuda").int().view(1, -1), i32([0, tokens]),
                                   i32([n]), i32(req), i32(row0), row_tiles, nq, nkv, d, page, n, 64 * waves if form == "decode" else 768, scale=1.0, waves=waves,
                                   tile_row1=None if row1 is None else i32(row1), grouped=grouped, even=waves > 1 and form != "decode").view(tokens, nq, d)
    scores = (k[:, 0, 0] + k[:, 0, 1]).double().expand(tokens, n).clone()
    scores[torch.arange(n, device="cuda")[None] > torch.arange(n - tokens, n, device="cuda")[:, None]] = -float("inf")
    want = torch.einsum("tk,khd->thd", scores.softmax(-1), v.double()).repeat_interleave(nq // nkv, 1)
    return out.double(), want


# products that climb slowly, quickly and far a step of keys; that fall; and that stand still
@pytest.mark.gpu
@pytest.mark.parametrize("climb", [0.02, 0.2, 0.3, 3.0, -0.5, 0.0])
@pytest.mark.parametrize("form", list(FORMS))
def test_a_rows_reference_follows_its_products(climb, form):
    """Key i has the product climb * i / log2(e) with every query, so the terms climb by 2^climb a key."""
    out, want = of_products(climb * torch.arange(700, device="cuda").float(), form)
    # weights rounded to bfloat16 (2^-8 of each, of values of up to five) and the result's own rounding
    assert bool(((out - want).abs() <= 2.0 ** -8 * want.abs() + 5 * 2.0 ** -8).all())
    assert float((out - want).norm() / want.norm()) <= 2.0 ** -8


@pytest.mark.gpu
@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("after", [40, 300])
def test_the_greatest_weight_is_not_rounded(form, after):
    """A key that outweighs all others, met behind one that is below it by a little or a lot: its weight is the reference's own, exactly one, so
    that the result has the rounding of bfloat16 and no other."""
    rows = torch.full((448,), -30.0, device="cuda")
    rows[3] = 0
    for above in torch.linspace(5.0, 9.0, 33).tolist():
        rows[after] = above
        out, want = of_products(rows, form)
        out, want = out[-1], want[-1]
        # the result's rounding; the other key's weight, 2^-above of the sum, rounded by 2^-8 of it (values of up to five); 32-bit sums
        assert bool(((out - want).abs() <= 2.0 ** -8 * want.abs() + 5 * 2.0 ** (-above - 8) + 5 * 2.0 ** -20).all()), above
