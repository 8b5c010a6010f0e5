"""Linear attention in chunks against the recurrence: numbers of chunks around those whose operands are on their way at a time, blocks of
columns shared out over several workgroups and over one, key heads of one slab to four."""

import pytest
import torch

from tokasaurus_amd.kernels import ops

pytestmark = pytest.mark.gpu


def plan(lengths, shortest=1):
    req, row0, first, at = [], [], [0], 0
    for r, n in enumerate(lengths):
        rows = range(at, at + n, ops.linear_attention_chunk_tokens()) if n >= shortest else ()
        req, row0, at = req + [r] * len(rows), row0 + list(rows), at + n
        first.append(len(req))
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    return ops.ChunkPlan(i32(req), i32(row0), i32(first), sum(n < shortest for n in lengths))


@pytest.mark.parametrize("heads,dk,dv,lengths", [(2, 128, 144, [64 * 4, 64 * 5 + 1, 64 * 6 - 1]), (1, 64, 16, [64 * 11]), (3, 200, 33, [33, 64 * 10]),
                                                 (1, 256, 130, [64 * 5, 1, 40]), (16, 20, 128, [64 * 3 + 7] * 9)])
@pytest.mark.parametrize("memory", [False, True])
def test_chunks_follow_the_recurrence(heads, dk, dv, lengths, memory):
    g = torch.Generator(device="cuda").manual_seed(dk + dv)
    rand = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    n, R, off = sum(lengths), len(lengths), heads * (2 * dk + dv)
    proj, before = rand(n, off + max(2 * heads, 16)), rand(R + 1, ops.linear_attention_state_words(heads, dk, dv, memory)) * 0.3
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    starts, slots = i32([sum(lengths[:i]) for i in range(R + 1)]), i32(range(R, 0, -1))
    up, bias, i_bias, f_bias = rand(16, heads * dk) * 0.3, rand(heads * dk), rand(heads), rand(heads) + 2

    def run(chunks):
        state = before.clone()
        if memory:
            positions = torch.cat([torch.arange(m) for m in lengths]).int().cuda()
            o, _ = ops.matrix_memory(proj, 0, heads * dk, 2 * heads * dk, off, off + heads, i_bias, f_bias, 15.0, dk ** -0.5, state, starts, slots,
                                     positions, heads, dk, dv, max(lengths), chunks=chunks)
            o = o.view(n, heads, -1)[..., : dv + 1]
        else:
            o = ops.gated_linear_attention(proj, 0, heads * dk, 2 * heads * dk, off, up, bias, 16.0, dk ** -0.5, state, starts, slots, heads, dk, dv,
                                           max(lengths), chunks=chunks)
        return o, state

    (o, state), (want_o, want_state) = run(plan(lengths)), run(None)
    rel = lambda x, y: float((x.double() - y.double()).norm() / y.double().norm())  # noqa: E731
    # the same terms in two orders: a decay's exponent is a sum of up to 64 logarithms of about one each in one of them (64 roundings of
    # 2^-24 of up to 64), a product of as many factors in the other
    assert rel(o, want_o) <= 64 * 2.0 ** -24 and rel(state[1:], want_state[1:]) <= 64 * 2.0 ** -24
    assert torch.equal(state[0], before[0])


@pytest.mark.parametrize("tau", [5.0, 15.0, 16.0])
def test_a_quotient_by_tau_is_not_off_to_one_side(tau):
    """One token's key and value behind 63 decays of a channel: the state is exp(63 log(sigmoid(bias)) / tau)."""
    g = torch.Generator(device="cuda").manual_seed(5)
    heads, dk, dv, n = 8, 256, 16, 64
    off = heads * (2 * dk + dv)
    proj = torch.zeros((n, off + 16), device="cuda")
    proj[0, heads * dk: off] = 1
    bias = torch.rand((heads * dk,), generator=g, device="cuda") * 2 - 1
    state = torch.zeros((2, ops.linear_attention_state_words(heads, dk, dv, False)), device="cuda")
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    ops.gated_linear_attention(proj, 0, heads * dk, 2 * heads * dk, off, torch.zeros((16, heads * dk), device="cuda"), bias, tau, 1.0, state, i32([0, n]), i32([1]),
                               heads, dk, dv, n, chunks=plan([n]))
    got, log_a = state[1].view(heads, dv, dk)[:, 0].double(), 63 * torch.nn.functional.logsigmoid(bias.double()).view(heads, dk) / tau
    off_by = (torch.log(got) - log_a) / log_a
    # the mean of 2,048 channels' errors, each a sum's of 64 terms and an exponential's (a few 2^-24 of the logarithm): a third of a rounding, where the
    # quotient rounded once is off by up to 2^-24
    assert abs(float(off_by.mean())) <= 2.0 ** -24 / 3


@pytest.mark.parametrize("heads,dk,dv,lengths", [(8, 128, 128, [70, 1, 200, 1, 1]), (2, 40, 24, [1, 64, 1]), (1, 256, 130, [33] + [1] * 40)])
@pytest.mark.parametrize("memory", [False, True])
def test_single_tokens_beside_chunks(heads, dk, dv, lengths, memory):
    """Requests of one token have the bits of a step of single tokens, the others those of a step without them."""
    g = torch.Generator(device="cuda").manual_seed(dk + len(lengths))
    rand = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    n, R, off = sum(lengths), len(lengths), heads * (2 * dk + dv)
    proj, before = rand(n, off + max(2 * heads, 16)), rand(R + 1, ops.linear_attention_state_words(heads, dk, dv, memory)) * 0.3
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    at = [sum(lengths[:i]) for i in range(R + 1)]
    up, bias, i_bias, f_bias = rand(16, heads * dk) * 0.3, rand(heads * dk), rand(heads), rand(heads) + 2
    past = [5 * r for r in range(R)]

    def run(which, chunks):
        rows = torch.cat([proj[at[r]: at[r + 1]] for r in which])
        some = [lengths[r] for r in which]
        starts, slots = i32([sum(some[:i]) for i in range(len(some) + 1)]), i32([R - r for r in which])
        state = before.clone()
        if memory:
            positions = torch.cat([torch.arange(past[r], past[r] + lengths[r]) for r in which]).int().cuda()
            o, floor = ops.matrix_memory(rows, 0, heads * dk, 2 * heads * dk, off, off + heads, i_bias, f_bias, 15.0, dk ** -0.5, state, starts, slots,
                                         positions, heads, dk, dv, max(some), chunks=chunks)
            o = torch.cat([o.view(len(rows), heads, -1)[..., : dv + 1].flatten(1), floor.view(len(rows), -1)], 1)
        else:
            o = ops.gated_linear_attention(rows, 0, heads * dk, 2 * heads * dk, off, up, bias, 16.0, dk ** -0.5, state, starts, slots, heads, dk, dv,
                                           max(some), chunks=chunks)
        return dict(zip(which, o.split(some))), state

    singles, others = [r for r in range(R) if lengths[r] == 1], [r for r in range(R) if lengths[r] > 1]
    both, state = run(list(range(R)), plan(lengths, shortest=2))
    one, state_one = run(singles, None)
    long, state_long = run(others, plan([lengths[r] for r in others]))
    for some, o, s in ((singles, one, state_one), (others, long, state_long)):
        for r in some:
            assert torch.equal(both[r], o[r]) and torch.equal(state[R - r], s[R - r]), r
    assert torch.equal(state[0], before[0])


def test_plans_of_a_step_leave_single_tokens_out():
    from test_parts_gpu import context
    from tokasaurus_amd.parts.linear_attention import chunk_plan

    ctx, _ = context([100, 40, 1, 1, 1], [0, 7, 3, 9, 20], [[0], [1], [2], [3], [4]], torch.bfloat16)
    for memory in (False, True):
        p = chunk_plan(ctx, memory, 128)
        lengths = [ctx.host_q_start[r + 1] - ctx.host_q_start[r] for r in range(5)]
        assert p.req.numel() == sum(-(-n // ops.linear_attention_chunk_tokens()) for n in lengths if n > 1) and p.without == 3
