"""Prompts in bfloat16 through the matrix-core attention of 32-bit arithmetic, one tile of 16 tokens a wavefront: steps of two
blocks of 16 keys, the weights in three exact bfloat16 pieces, tiles dealt to the workgroups by length.  Against sums in
64-bit."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _paged(lens, nkv, dk, dv, page, gen):
    """Keys and values of requests of these lengths, in pages in shuffled order; every place behind a request's end is NaN."""
    pages = [-(-n // page) for n in lens]
    order = (torch.randperm(sum(pages), generator=gen) + 1).tolist()
    table = torch.zeros((len(lens), max(pages)), dtype=torch.int32)
    kc = torch.full((sum(pages) + 1, nkv, dk // 8, page, 8), float("nan"), dtype=torch.bfloat16)
    vc = torch.full((sum(pages) + 1, nkv, page // 4, dv, 4), float("nan"), dtype=torch.bfloat16)
    keys = [torch.randn((n, nkv, dk), generator=gen).bfloat16() for n in lens]
    values = [torch.randn((n, nkv, dv), generator=gen).bfloat16() for n in lens]
    for r, n in enumerate(lens):
        for i in range(pages[r]):
            p = table[r, i] = order.pop()
            m = min(page, n - i * page)
            k = torch.full((page, nkv, dk), float("nan"), dtype=torch.bfloat16)
            v = torch.full((page, nkv, dv), float("nan"), dtype=torch.bfloat16)
            k[:m], v[:m] = keys[r][i * page: i * page + m], values[r][i * page: i * page + m]
            kc[p] = k.view(page, nkv, dk // 8, 8).permute(1, 2, 0, 3)
            vc[p] = v.view(page // 4, 4, nkv, dv).permute(2, 0, 3, 1)
    return keys, values, kc, vc, table


def _run(q, kc, vc, table, portions, lens, nq, nkv, dk, dv, page, **options):
    from tokasaurus_amd.kernels import ops

    start = [0]
    for n in portions:
        start.append(start[-1] + n)
    tiles = [(r, a) for r in range(len(lens)) for a in range(start[r], start[r + 1], 16)]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    out = ops.attention_tile_f32(q.cuda().view(start[-1], nq * dk), kc.cuda(), vc.cuda(), table.cuda(), i32(start), i32(lens),
                                 i32([r for r, _ in tiles]), i32([a for _, a in tiles]), nq, nkv, dk, dv, page, 1, **options)
    return out.cpu().view(start[-1], nq, dv), start


@pytest.mark.parametrize("lens,portions,nq,nkv,dk,dv,page,options", [
    ([1], [1], 2, 1, 8, 16, 16, {}),
    ([31, 32, 33], [31, 32, 33], 8, 2, 64, 64, 16, {}),  # the second block of a step in another page, or beyond the end
    ([17, 300], [17, 40], 4, 2, 40, 48, 48, {}),  # a later portion of a prompt; sizes that fill no block
    ([200], [200], 4, 4, 64, 32, 16, {"window": 40}),
    ([200], [200], 4, 1, 32, 64, 64, {"section": 50}),
    ([150], [150], 8, 8, 128, 128, 32, {"softcap": 5.0}),
    ([150], [150], 4, 2, 64, 64, 32, {"score_bias": True}),
    ([40], [40], 2, 2, 256, 256, 16, {}),  # heads too wide for two blocks a step
    ([700, 65], [700, 65], 32, 8, 64, 64, 64, {}),  # 49 tiles x 8 workgroups: one round of 256 and a part of the next
    ([400, 900], [400, 900], 28, 4, 64, 64, 64, {}),  # 82 tiles x 7: rounds in both directions, heads that leave wavefronts idle
])
def test_prompts_against_64_bit_sums(lens, portions, nq, nkv, dk, dv, page, options):
    gen = torch.Generator().manual_seed(sum(lens) + dk)
    keys, values, kc, vc, table = _paged(lens, nkv, dk, dv, page, gen)
    q = torch.randn((sum(portions), nq, dk), generator=gen).bfloat16()
    bias = torch.randn((nq,), generator=gen) if options.get("score_bias") else None
    given = dict(options, **({"score_bias": bias.cuda()} if bias is not None else {}))
    scale = dk ** -0.5
    out, start = _run(q, kc, vc, table, portions, lens, nq, nkv, dk, dv, page, scale=scale, split=False, **given)
    for r, n in enumerate(lens):
        Q = q[start[r]: start[r + 1]].double()
        K = keys[r].double().repeat_interleave(nq // nkv, 1)
        V = values[r].double().repeat_interleave(nq // nkv, 1)
        s = torch.einsum("thd,khd->htk", Q, K) * float(torch.tensor(scale, dtype=torch.float32))
        if "softcap" in options:
            s = options["softcap"] * torch.tanh(s / options["softcap"])
        pos = torch.arange(n - portions[r], n)[:, None]
        key = torch.arange(n)[None]
        seen = key <= pos
        if "window" in options:
            seen = seen & (pos - key < options["window"])
        if "section" in options:
            seen = seen & (pos // options["section"] == key // options["section"])
        if bias is None:
            w = torch.softmax(s.masked_fill(~seen, float("-inf")), -1)
        else:
            w = torch.sigmoid(s + bias.double()[:, None, None]) * seen
        want = torch.einsum("htk,khd->thd", w, V)
        # the result is rounded once to bfloat16 (8 bits: up to 2^-8 of it); scores are 32-bit sums of dk products (their error moves
        # a weight by as much, relatively), and the sums over the keys 32-bit sums of n
        size = torch.einsum("htk,khd->thd", w, V.abs())
        reach = float((torch.einsum("thd,khd->htk", Q.abs(), K.abs()) * scale).max())
        limit = want.abs() * 2.0 ** -8 + size * (n + 64 + dk * reach) * 2.0 ** -23
        assert ((out[start[r]: start[r + 1]].double() - want).abs() <= limit).all()


def test_infinite_values_stay_infinite():
    """A value that is infinite meets a weight's pieces that are zero: the sum must be what the 32-bit product gives."""
    gen = torch.Generator().manual_seed(5)
    n, page = 130, 16
    keys, values, kc, vc, table = _paged([n], 1, 64, 64, page, gen)
    at = 37
    vc[table[0, at // page], 0, at % page // 4, 3, at % 4] = float("inf")
    vc[table[0, at // page], 0, at % page // 4, 5, at % 4] = float("-inf")
    q = torch.randn((n, 2, 64), generator=gen).bfloat16()
    out, _ = _run(q, kc, vc, table, [n], [n], 2, 1, 64, 64, page, scale=0.125, split=False)
    both, _ = _run(q, kc, vc, table, [n], [n], 2, 1, 64, 64, page, scale=0.125, split=True)  # 32-bit products
    assert (out[48:, :, 3] == float("inf")).all() and (out[48:, :, 5] == float("-inf")).all()
    assert torch.isfinite(out[:32]).all()
    assert torch.equal(torch.isfinite(out), torch.isfinite(both)) and torch.equal(torch.isnan(out), torch.isnan(both))


def test_which_prompts_take_a_tile_a_wavefront():
    """With the step's longest request given, bfloat16 prompts leave the split form from 512 pairs on; single tokens do not."""
    gen = torch.Generator().manual_seed(9)
    lens = [300]
    keys, values, kc, vc, table = _paged(lens, 8, 64, 64, 64, gen)
    q = torch.randn((300, 32, 64), generator=gen).bfloat16()
    args = (q, kc, vc, table, lens, lens, 32, 8, 64, 64, 64)
    chosen, _ = _run(*args, longest=300)
    plain, _ = _run(*args, split=False)
    split, _ = _run(*args, split=True)
    assert torch.equal(chosen, plain)
    unknown, _ = _run(*args)  # 608 pairs, nothing known of the lengths
    assert torch.equal(unknown, split)


def test_an_engines_prompt_takes_a_tile_a_wavefront(tmp_path, monkeypatch):
    """Through the runner with its default planning bound (1,024 keys), which says nothing of the step's own lengths."""
    from kupuzen_models import TOL, attention_layer, compare_rows, make_folder, plain_rows
    from tokasaurus_amd.engine.batch import StepEntry
    from tokasaurus_amd.engine.runner import ModelRunner
    from tokasaurus_amd.kernels import ops

    cfg = {"architecture": "Kupuzen", "vocab": 120, "width": 64, "embedding": {"scale": 2.0}, "norm": {"eps": 1e-5}, "residual_mult": 0.7,
           "layers": [attention_layer(32, 2, 8, 16, 0.3, rot={"base": 100.0, "dims": 8})]}
    folder = make_folder(tmp_path / "wide", cfg, seed=4)
    runner = ModelRunner.from_folder(str(folder), "bfloat16", page_size=16, num_pages=160, max_slots=4)
    assert runner.kv_bound(260) == 1024
    chosen = []
    rule = ops.attention_tile_splits
    monkeypatch.setattr(ops, "attention_tile_splits", lambda *a, **kw: chosen.append(rule(*a, **kw)) or chosen[-1])
    tokens = [(7 * i + 3) % 120 for i in range(300)]
    out = runner.run([StepEntry("a", tokens[:260], [259])])
    assert chosen == [False]  # 17 tiles x 32 heads
    got = {("a", 259): out.logits[0].float().cpu()}
    runner.run([StepEntry("a", tokens[260:290], [])])  # after a past longer than the step: shared tiles
    runner.run([StepEntry("a", tokens[290:291], [])])
    assert len(chosen) >= 3 and all(chosen[1:])
    compare_rows(got, plain_rows(folder, {"a": tokens}), TOL["bfloat16"])


@pytest.mark.parametrize("options", [{}, {"window": 100}, {"section": 150}])
def test_chunks_end_with_the_steps_own_longest_request(options):
    """The chunks behind it hold nothing: without them the sums are the same, bit by bit."""
    gen = torch.Generator().manual_seed(11)
    lens, portions = [200, 1100], [16, 40]
    keys, values, kc, vc, table = _paged(lens, 2, 64, 64, 16, gen)
    q = torch.randn((sum(portions), 4, 64), generator=gen).bfloat16()
    args = (q, kc, vc, table, portions, lens, 4, 2, 64, 64, 16)
    planned, _ = _run(*args, split=True, key_chunk=256, longest=8192, scale=0.125, **options)
    own, _ = _run(*args, split=True, key_chunk=256, longest=8192, step_longest=1100, scale=0.125, **options)
    assert torch.isfinite(own).all() and torch.equal(own, planned)


@pytest.mark.parametrize("dk,dv", [(64, 64), (128, 128), (24, 176)])  # (176: heads of one block a step)
@pytest.mark.parametrize("slope", [-0.4, 0.0, 0.01, 0.4, 4.0])
@pytest.mark.parametrize("softcap", [0.0, 200.0, 30.0])
def test_scores_that_rise_and_sinks(dk, dv, slope, softcap):
    """Scores that rise with the keys by less than a reference allows, or by more (and fall), tanh on both sides of where its
    polynomial ends, and sinks below, near and far above all of them."""
    gen = torch.Generator().manual_seed(dk + int(100 * slope))
    n, nq, nkv, page = 100, 4, 1, 16
    keys, values, kc, vc, table = _paged([n], nkv, dk, dv, page, gen)
    keys[0][:, :, 0] = (torch.arange(n) * slope).bfloat16()[:, None]
    for i in range(-(-n // page)):
        m = min(page, n - i * page)
        kc[table[0, i], :, 0, :m, 0] = keys[0][i * page: i * page + m, :, 0].T
    q = torch.randn((n, nq, dk), generator=gen).bfloat16()
    q[:, :, 0] = dk ** 0.5
    sink = torch.tensor([-1000.0, 0.0, 40.0, 1000.0])
    options = {"softcap": softcap} if softcap else {}
    out, _ = _run(q, kc, vc, table, [n], [n], nq, nkv, dk, dv, page, scale=dk ** -0.5, split=False, sink=sink.cuda(), **options)
    s = torch.einsum("thd,kd->htk", q.double(), keys[0][:, 0].double()) * float(torch.tensor(dk ** -0.5, dtype=torch.float32))
    if softcap:
        s = softcap * torch.tanh(s / softcap)
    s = s.masked_fill(torch.ones((n, n)).triu(1).bool(), -float("inf"))
    p = torch.softmax(torch.cat([s, sink.double()[:, None, None].expand(nq, n, 1)], -1), -1)[:, :, :n]
    want = torch.einsum("htk,kd->thd", p, values[0][:, 0].double())
    # the result's rounding (half a unit of 8 bits: 2^-8 of it), and of every weight that of its score (2^-24 of up to 400, scaled and in units of log 2) and of its exponential
    size = torch.einsum("htk,kd->thd", p, values[0][:, 0].double().abs())
    assert bool(((out.double() - want).abs() <= want.abs() * 2.0 ** -8 + size * 8 * 400 * 2.0 ** -24 + 1e-30).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("split", [False, True])
def test_capped_scores_depend_on_no_key_that_is_not_seen(dtype, split):
    """The places behind a request's end, and the page of no request, hold zeros, numbers far beyond the cap, or NaN: the same bits.
    (Scores of three to six tenths of the cap, where the ways to a tanh differ in their last bits.)"""
    gen = torch.Generator().manual_seed(12)
    lens, nq, nkv, d, page = [23, 70, 130], 4, 2, 64, 16
    _, _, kc, vc, table = _paged(lens, nkv, d, d, page, gen)
    scores = torch.zeros_like(kc)
    scores[:, :, 0, :, 0] = torch.rand(kc.shape[0], nkv, page, generator=gen) * 6 + 6
    kc = torch.where(kc.isnan(), kc, scores)
    q = torch.zeros((sum(lens), nq, d), dtype=dtype)
    q[:, :, 0] = 8
    got = []
    for stale in (0.0, 1e4, -1e4, float("nan")):
        k, v = (torch.where(x.isnan(), torch.tensor(stale, dtype=x.dtype), x).to(dtype) for x in (kc, vc))
        out, _ = _run(q, k, v, table, lens, lens, nq, nkv, d, d, page, scale=d ** -0.5, split=split, softcap=20.0)
        got.append(out)
    assert torch.isfinite(got[0]).all() and all(torch.equal(x, got[0]) for x in got[1:])


@pytest.mark.parametrize("split", [False, True])
def test_capped_scores_have_no_error_but_their_rounding(split):
    """Tokens that see themselves alone beside a sink that is near their score, so that the weight shows a score's error: exact products over a cap of
    32, tanh of a half to five eighths."""
    gen = torch.Generator().manual_seed(13)
    n, d, page, cap, sink = 16384, 16, 64, 32.0, 16.25
    x = (torch.rand((n,), generator=gen) / 8 + 0.5) * cap
    kc, vc = torch.zeros((n // page, 1, d // 8, page, 8)), torch.ones((n // page, 1, page // 4, d, 4))
    kc[:, 0, 0, :, 0] = x.view(-1, page)
    q = torch.zeros((n, 1, d))
    q[:, :, 0] = 1
    table = torch.arange(n // page, dtype=torch.int32)[None]
    out, _ = _run(q, kc, vc, table, [n], [n], 1, 1, d, d, page, scale=1.0, softcap=cap, section=1, sink=torch.tensor([sink]).cuda(), split=split)
    w, score = out[:, 0, 0].double(), cap * torch.tanh(x.double() / cap)
    off = (torch.log(w / (1 - w)) + sink - score) / score
    # the mean of the roundings (6e-8 at most each of the tanh, of the score and of the weight's terms, root mean square of all 4e-8) over 16,384, eight times as much
    assert abs(float(off.mean())) <= 2.5e-9
    assert float(off.pow(2).mean().sqrt()) <= 6e-8


@pytest.mark.parametrize("product,value", [(5.0, 3e38), (2.5e38, 1.0), (-2.5e38, 1.0)])
def test_sums_that_are_finite_by_weights_of_one_and_less(product, value):
    """A key whose values are near the largest numbers and whose score is above the others' by less than a reference lags behind; scores whose
    product with log2(e) is beyond 32 bits: against 64 bits, with and without a sink far below."""
    gen = torch.Generator().manual_seed(14)
    n, at, d, page = 40, 33, 64, 16
    keys, values, kc, vc, table = _paged([n], 1, d, d, page, gen)
    side = abs(product) ** 0.5
    keys[0][:] = 0
    keys[0][:, 0, 0] = -side if product < -9 else 0  # (all others are lowest where the one is greatest)
    keys[0][at, 0, 0] = side if product > 0 else -side / 2
    values[0][at] = (values[0][at].sign().float() * value).bfloat16()
    for p in range(-(-n // page)):
        m = min(page, n - p * page)
        kc[table[0, p], 0, :, :m] = keys[0][p * page: p * page + m, 0].view(m, d // 8, 8).permute(1, 0, 2)
    vc[table[0, at // page], 0, at % page // 4, :, at % 4] = values[0][at, 0]
    q = torch.zeros((n, 2, d), dtype=torch.bfloat16)
    q[:, :, 0] = side
    s = torch.einsum("thd,kd->htk", q.double(), keys[0][:, 0].double()).masked_fill(torch.ones((n, n)).triu(1).bool(), -float("inf"))
    w = torch.softmax(s, -1)
    want = torch.einsum("htk,kd->thd", w, values[0][:, 0].double())
    size = torch.einsum("htk,kd->thd", w, values[0][:, 0].double().abs())
    for sink in (None, torch.full((2,), -3.3e38).cuda()):
        out, _ = _run(q, kc, vc, table, [n], [n], 2, 1, d, d, page, scale=1.0, split=False, sink=sink)
        assert bool(((out.double() - want).abs() <= want.abs() * 2.0 ** -8 + size * n * 2.0 ** -22).all()), sink
