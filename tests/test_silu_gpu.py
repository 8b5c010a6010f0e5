"""The activation of gate and up in bfloat16, for every number there is."""

import pytest
import torch

from tokasaurus_amd.kernels import ops

pytestmark = pytest.mark.gpu


def test_every_gate_is_rounded_to_the_nearest():
    gate = torch.arange(-32768, 32768, dtype=torch.int32).to(torch.int16).view(torch.bfloat16).view(64, 1024)
    got = ops.swiglu(torch.cat([gate, torch.ones_like(gate)], 1).cuda()).cpu().double()
    x = gate.double()
    want = x / (1 + torch.exp(-x))
    # exp(-x) is past the 32-bit numbers there: -0 (and of minus infinity nothing)
    past = x < -88.7
    assert bool((got[past & torch.isfinite(x)] == 0).all()) and bool(torch.isnan(got[torch.isnan(x) | (x == -float("inf"))]).all())
    assert float(got[x == float("inf")]) == float("inf")
    rest = torch.isfinite(x) & ~past
    # half of a bfloat16 number's last place, and where the quotient falls into the middle of two its 32 bits decide (four roundings of
    # 2^-24, and |x| times one in the exponent: below 2^-15 in all)
    half = torch.ldexp(torch.ones_like(want), want.abs().log2().floor().clamp_min(-126) - 8)
    worst = ((got - want).abs() / (half + 2.0 ** -15 * want.abs() + 1e-300))[rest]
    assert float(worst.max()) <= 1.0
