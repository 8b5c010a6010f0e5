"""The activation of gate and up in bfloat16, for every number there is: of the kernel behind a product, and of the products that have it in
their own kernels, which compute it another way."""

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


def _gated(x, w, kernel):
    if kernel == "tiles":
        return ops.gemm_tiles_bf16(x, w, 0, glu=True)
    return ops.gemm_skinny_bf16(x, w, swiglu=True, staged=2 if kernel == "streamed" else 0)


def _same(got, want):
    numbers = ~torch.isnan(want)
    return torch.equal(torch.isnan(got), ~numbers) and torch.equal(got[numbers].view(torch.int16), want[numbers].view(torch.int16))


@pytest.mark.parametrize("kernel", ["few rows", "streamed", "tiles"])
def test_every_gate_in_a_product_has_the_bits_of_the_division(kernel):
    """Rows of x that are one in one place and zero elsewhere: a gate is a number of the weight, its up is 1.  What the product's own kernel makes
    of it is then, bit for bit, what x / (1 + expf(-x)) gives, computed in 32 bits by the pass behind a product and rounded."""
    k = 64
    x = torch.eye(k, dtype=torch.bfloat16).cuda()
    every = torch.arange(-32768, 32768, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    finite = torch.where(torch.isfinite(every), every, torch.zeros_like(every)).view(1024, k).cuda()
    w = torch.cat([finite, torch.ones_like(finite)])
    gate = finite.t().contiguous() + 0.0  # (a sum of zeros is +0)
    want = ops.swiglu(torch.cat([gate, torch.ones_like(gate)], 1).float()).to(torch.bfloat16)
    assert _same(_gated(x, w, kernel), want)
    # infinities and no numbers by themselves: beside a zero of x they would be no numbers everywhere
    others = torch.zeros((1024, k), dtype=torch.bfloat16)
    odd = every[~torch.isfinite(every)]
    others[:, 0] = odd.repeat(1024 // odd.numel() + 1)[:1024]
    others = others.cuda()
    got = _gated(torch.ones((k, k), dtype=torch.bfloat16).cuda(), torch.cat([others, torch.full_like(others, 1.0 / k)]), kernel)
    gate = others[:, 0].expand(k, 1024).contiguous()
    want = ops.swiglu(torch.cat([gate, torch.ones_like(gate)], 1).float()).to(torch.bfloat16)
    assert _same(got, want)
