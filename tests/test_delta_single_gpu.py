"""A step of single tokens through the delta rule in one kernel: the bits of the three kernels that it stands for."""

import pytest
import torch

from tokasaurus_amd.kernels import ops

pytestmark = pytest.mark.gpu


# heads of one lane's pieces and of four, columns of one, two and four a thread, tails of none, three (the unrolled case) and more
@pytest.mark.parametrize("heads,dk,dv,taps", [(2, 128, 128, 4), (4, 16, 8, 3), (3, 100, 40, 1), (1, 256, 256, 4), (2, 64, 72, 5), (1, 4, 200, 2), (2, 132, 130, 4)])
@pytest.mark.parametrize("requests", [1, 5])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_one_kernel_has_the_bits_of_three(heads, dk, dv, taps, requests, dtype):
    g = torch.Generator(device="cuda").manual_seed(dk + dv + requests)
    rand = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    n, C = requests, heads * (2 * dk + dv)
    proj = rand(n, C + heads + 5).to(dtype)
    low = rand(n, heads * (dk + dv))
    a_pre, gate = low[:, : heads * dk], low[:, heads * dk:]
    conv_w, a_log, dt_bias, weight = rand(C, taps) * 0.5, rand(heads) * 0.5, rand(heads * dk) * 0.5, 1 + 0.1 * rand(dv)
    before = rand(n + 2, -(-ops.delta_state_size(heads, heads, dk, dv, taps) // 4) * 4) * 0.3
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    starts, slots = i32(range(n + 1)), i32(range(n, 0, -1))
    args = (proj, C + 2, a_pre, conv_w, a_log, dt_bias)
    three = before.clone()
    rec = ops.delta_prepare(*args, three, starts, i32(range(n)), slots, heads, heads, dk, dv)
    want = ops.gated_head_norm(ops.delta_rule(rec, three, starts, slots, heads, heads, dk, dv), gate, weight, 1e-6, heads, dv, dtype)
    one = before.clone()
    assert ops.delta_single_takes(n, slots, heads, heads, dk, dv, one)
    got = ops.delta_single(*args, one, starts, slots, gate, weight, 1e-6, heads, dk, dv, dtype)
    assert torch.equal(got, want) and torch.equal(one, three)


def test_what_it_leaves_to_the_three_kernels():
    state, slots = torch.zeros(3, 4096, device="cuda"), torch.zeros(2, dtype=torch.int32, device="cuda")
    assert ops.delta_single_takes(2, slots, 2, 2, 16, 8, state)
    for tokens, heads, groups, dk, dv in ((3, 2, 2, 16, 8), (2, 2, 1, 16, 8), (2, 2, 2, 18, 8), (2, 1, 1, 260, 8), (2, 1, 1, 4, 260)):
        assert not ops.delta_single_takes(tokens, slots, heads, groups, dk, dv, state)
    assert not ops.delta_single_takes(2, slots, 2, 2, 16, 8, torch.zeros(3, 4098, device="cuda"))
