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
