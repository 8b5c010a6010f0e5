"""Decays exp(-softplus(x)) of the delta rule against 64 bits: no further off than a softplus by the logarithm and exponential of the
mathematics library, whose own errors over the same numbers are the bounds."""

import pytest
import torch

from tokasaurus_amd.kernels import ops

pytestmark = pytest.mark.gpu


def decays(x):
    """x [tokens, 256] through the kernel that prepares the delta rule's rows: one head, a rate of one."""
    n, d = x.shape
    zeros = lambda *s: torch.zeros(s, device="cuda")  # noqa: E731
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    rec = ops.delta_prepare(zeros(n, 2 * d + 16 + 1), 2 * d + 16, x, zeros(2 * d + 16, 2), zeros(1), zeros(d), zeros(1, d * 16 + 2 * d + 16), i32([0, n]),
                            i32([0] * n), i32([0]), 1, 1, d, 16)
    return rec[:, 2 * d + 16: 3 * d + 16]


@pytest.mark.parametrize("reach,rms,largest", [(2.0, 1.64e-8, 7.4e-8), (12.0, 1.357e-8, 7.4e-8)])
def test_decays_are_as_near_as_the_librarys(reach, rms, largest):
    n = 16384 * 256
    x = ((torch.arange(n, dtype=torch.float64) + 0.5) / n * 2 - 1).mul(reach).float().view(-1, 256).cuda()
    off = decays(x).double() - torch.sigmoid(-x.double())
    assert float(off.pow(2).mean().sqrt()) <= rms and float(off.abs().max()) <= largest


def test_softplus_at_its_ends():
    x = torch.tensor([float("inf"), -float("inf"), float("nan"), 90.0, -90.0, 64.0, 3e38, -3e38, 0.0, 1e-30], device="cuda")
    got = decays(x[:, None].expand(-1, 256).contiguous())[:, 7].cpu()
    assert torch.isnan(got[2]) and got[0] == 0 and got[6] == 0 and got[1] == 1 and got[4] == 1 and got[7] == 1
    assert got[8] == 0.5 and got[9] == 0.5 and abs(float(got[3]) / 8.194e-40 - 1) < 1e-3 and abs(float(got[5]) / 1.6038e-28 - 1) < 1e-4
