"""The delta rule in chunks against the recurrence in 64 bits, and against the recurrence's own kernel: sizes that fill no block,
chunks that end early, requests of every length in a step, states and tails from before, decays near one and near zero."""

import pytest
import torch

from tokasaurus_amd.kernels import ops

pytestmark = pytest.mark.gpu


def reference(proj, col_b, a_pre, conv_w, a_log, dt_bias, state, starts, slots, H, G, dk, dv):
    """(o, state) in 64 bits, token by token."""
    d = lambda t: t.double()  # noqa: E731
    proj, a_pre, conv_w, state = d(proj), d(a_pre), d(conv_w), d(state).clone()
    C, taps = conv_w.shape
    o = torch.zeros((proj.shape[0], H, dv), dtype=torch.float64, device=proj.device)
    tail_at = H * dk * dv
    for r, slot in enumerate(slots):
        a, b = starts[r], starts[r + 1]
        tail = state[slot, tail_at : tail_at + (taps - 1) * C].view(taps - 1, C)
        rows = torch.cat([tail, proj[a:b, :C]])
        y = sum(rows[j : j + b - a] * conv_w[:, j] for j in range(taps))
        y = y * torch.sigmoid(y)
        q, k = (y[:, i * G * dk : (i + 1) * G * dk].view(-1, G, dk).repeat_interleave(H // G, 1) for i in range(2))
        v = y[:, 2 * G * dk :].view(-1, H, dv)
        unit = lambda x: x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
        q, k = unit(q) * dk ** -0.5, unit(k)
        g = torch.exp(-torch.exp(d(a_log))[:, None] * torch.nn.functional.softplus((a_pre[a:b] + d(dt_bias)).view(-1, H, dk)))
        beta = torch.sigmoid(proj[a:b, col_b : col_b + H])
        S = state[slot, :tail_at].view(H, dv, dk).transpose(1, 2).clone()
        for t in range(b - a):
            S = g[t][..., None] * S
            u = beta[t][:, None] * (v[t] - (k[t][:, None] @ S)[:, 0])
            S = S + k[t][..., None] * u[:, None]
            o[a + t] = (q[t][:, None] @ S)[:, 0]
        state[slot, :tail_at] = S.transpose(1, 2).reshape(-1)
        state[slot, tail_at : tail_at + (taps - 1) * C] = rows[b - a :].reshape(-1)
    return o.flatten(1), state


def cut(starts, size):
    req, row0, first = [], [], [0]
    for r in range(len(starts) - 1):
        rows = range(starts[r], starts[r + 1], size)
        req, row0 = req + [r] * len(rows), row0 + list(rows)
        first.append(len(req))
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    return ops.ChunkPlan(i32(req), i32(row0), i32(first))


@pytest.mark.parametrize("heads,groups,dk,dv,taps", [(2, 2, 128, 128, 4), (4, 2, 16, 8, 3), (3, 1, 100, 40, 1), (2, 1, 64, 72, 5), (1, 1, 256, 256, 4)])
@pytest.mark.parametrize("lengths", [[32], [47, 16, 33, 1], [17, 150]])
@pytest.mark.parametrize("decay", [-4.0, 0.0, 3.0])  # decays of about 0.98, 0.5 and 1e-6
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_chunks_follow_the_recurrence(heads, groups, dk, dv, taps, lengths, decay, dtype):
    g = torch.Generator(device="cuda").manual_seed(dk + dv + sum(lengths))
    rand = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    n, C = sum(lengths), 2 * groups * dk + heads * dv
    starts = [sum(lengths[:i]) for i in range(len(lengths) + 1)]
    size = ops.delta_chunk_tokens(dk, dv, max(lengths))
    assert size == 16
    proj = rand(n, C + heads + 5).to(dtype)
    a_pre, conv_w, a_log, dt_bias = rand(n, heads * dk + 3)[:, : heads * dk], rand(C, taps) * 0.5, rand(heads) * 0.5, rand(heads * dk) * 0.5 + decay
    words = ops.delta_state_size(heads, groups, dk, dv, taps)
    before = rand(len(lengths) + 2, words) * 0.3
    slots = list(range(len(lengths), 0, -1))
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    args = (proj, C + 2, a_pre, conv_w, a_log, dt_bias)
    want_o, want_s = reference(*args, before, starts, slots, heads, groups, dk, dv)
    state = before.clone()
    o = ops.delta_rule_chunks(*args, state, i32(starts), i32(slots), cut(starts, size), heads, groups, dk, dv)
    plain_state = before.clone()
    req = i32([r for r, m in enumerate(lengths) for _ in range(m)])
    rec = ops.delta_prepare(*args, plain_state, i32(starts), req, i32(slots), heads, groups, dk, dv)
    plain = ops.delta_rule(rec, plain_state, i32(starts), i32(slots), heads, groups, dk, dv)
    rel = lambda x, y: float((x.double() - y).norm() / y.norm())  # noqa: E731
    # both are 32-bit sums of the same terms in other orders: no further from the 64-bit ones than the recurrence's kernel
    # but for a factor, or than a few roundings
    for got, base, want in ((o, plain, want_o), (state, plain_state, want_s)):
        print(f"dk {dk} {lengths} decay {decay}: {rel(got, want):.2e}, recurrence {rel(base, want):.2e}")
        assert rel(got, want) <= max(1.5 * rel(base, want), 4 * 2.0 ** -24)
    untouched = [s for s in range(before.shape[0]) if s not in slots]
    assert torch.equal(state[untouched], before[untouched])
    tails = heads * dk * dv
    assert torch.equal(state[:, tails:], plain_state[:, tails:])


@pytest.mark.parametrize("lengths", [[40, 5, 100, 1, 31, 1], [1, 32], [33, 1, 1, 1], [31, 64]])
@pytest.mark.parametrize("heads,groups,dk,dv,taps", [(2, 1, 64, 72, 4), (2, 2, 20, 8, 1), (1, 1, 128, 128, 6)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_what_a_request_shares_its_step_with_changes_nothing(lengths, heads, groups, dk, dv, taps, dtype):
    """Requests of few tokens have the recurrence's bits, those of many the chunks', whoever shares the step."""
    g = torch.Generator(device="cuda").manual_seed(sum(lengths) + dk)
    rand = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    n, C, least = sum(lengths), 2 * groups * dk + heads * dv, ops.DELTA_CHUNKS_FROM
    starts = [sum(lengths[:i]) for i in range(len(lengths) + 1)]
    proj = rand(n, C + heads).to(dtype)
    a_pre, conv_w, a_log, dt_bias = rand(n, heads * dk), rand(C, taps) * 0.5, rand(heads) * 0.5, rand(heads * dk) * 0.5
    before = rand(len(lengths) + 1, ops.delta_state_size(heads, groups, dk, dv, taps)) * 0.3
    slots = list(range(len(lengths), 0, -1))
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    args, sizes = (proj, C, a_pre, conv_w, a_log, dt_bias), (heads, groups, dk, dv)
    req = i32([r for r, m in enumerate(lengths) for _ in range(m)])
    one, two, both = before.clone(), before.clone(), before.clone()
    chunked = ops.delta_rule_chunks(*args, one, i32(starts), i32(slots), cut(starts, 16), *sizes)
    plain = ops.delta_rule(ops.delta_prepare(*args, two, i32(starts), req, i32(slots), *sizes), two, i32(starts), i32(slots), *sizes)
    all_chunks = cut(starts, 16)
    keep = [i for i, r in enumerate(all_chunks.req.tolist()) if lengths[r] >= least]
    counts = [-(-m // 16) if m >= least else 0 for m in lengths]
    plan = ops.ChunkPlan(all_chunks.req[keep].contiguous(), all_chunks.row0[keep].contiguous(),
                         i32([sum(counts[:i]) for i in range(len(counts) + 1)]))
    few = next((r, starts[r]) for r, m in enumerate(lengths) if m < least)
    got = ops.delta_rule_chunks(*args, both, i32(starts), i32(slots), plan, *sizes, req, least, few)
    for r, m in enumerate(lengths):
        rows, slot = slice(starts[r], starts[r + 1]), slots[r]
        want, state = (chunked, one) if m >= least else (plain, two)
        assert torch.equal(got[rows], want[rows]) and torch.equal(both[slot], state[slot]), r
    assert torch.equal(both[0], before[0])


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_a_model_step_of_both_kinds_of_requests(tmp_path, dtype):
    from kupuzen_models import TOL, compare_rows, delta_layer, make_folder, plain_rows
    from tokasaurus_amd.engine.batch import StepEntry
    from tokasaurus_amd.engine.runner import ModelRunner

    cfg = {"architecture": "Kupuzen", "vocab": 120, "width": 64, "embedding": {"scale": 2.0}, "norm": {"eps": 1e-5}, "residual_mult": 0.7,
           "layers": [delta_layer(4, 2, 16, 24, 4, 8, 8), delta_layer(2, 2, 16, 16, 4, 8, 8)]}
    folder = make_folder(tmp_path / "delta", cfg, seed=6)
    tokens = {r: [(k * i + 3) % 120 for i in range(230)] for r, k in (("a", 7), ("b", 11), ("c", 13))}
    runner = ModelRunner.from_folder(str(folder), dtype, page_size=16, num_pages=64, max_slots=4)
    at, got = {r: 0 for r in tokens}, {}
    for step in ({"a": 40}, {"a": 1, "b": 170, "c": 20}, {"a": 150, "b": 1, "c": 34}, {"a": 1, "b": 2, "c": 1}):
        entries = [StepEntry(r, tokens[r][at[r] : at[r] + n], list(range(n))) for r, n in step.items()]
        rows = runner.run(entries).logits.float().cpu()
        places = [(r, at[r] + i) for r, n in step.items() for i in range(n)]
        got.update(zip(places, rows))
        at = {r: at[r] + step.get(r, 0) for r in at}
    compare_rows(got, plain_rows(folder, tokens), TOL[dtype])
