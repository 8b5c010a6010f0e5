"""The 32-bit product of few rows with the activation, or the rotation and append, in its kernel: the bits of the product and of the
kernel behind it, where the product sums in the same order, else within what two orders may differ by."""

import pytest
import torch

from tokasaurus_amd.kernels import ops
from tokasaurus_amd.kernels.library import KernelError
from tokasaurus_amd.kernels.ops import RopeAppend

pytestmark = pytest.mark.gpu


def draw(seed, *shapes):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn(s, generator=g, device="cuda") for s in shapes]


def same_order(m, n, k):
    """Whether the plain product has 16 weight rows a workgroup, as these have (``tk_gemm_f32``: 8 for few rows and a small weight)."""
    return m > 8 or n > 2048 or k % 32 or k < 256


# one wavefront, four and eight; K that ends inside a block; gates beyond the last workgroup's
@pytest.mark.parametrize("m", [1, 4, 9, 16])
@pytest.mark.parametrize("nk", [(1, 12), (14, 64), (48, 260), (260, 288), (1034, 4100)])
def test_gate_and_up(m, nk):
    n, k = nk
    x, w, bias = draw(m + n + k, (m, k + 4), (2 * n, k), (2 * n,))
    x, w = x[:, 4:], w * k ** -0.5
    for b in (None, bias):
        both = ops.gemm_generic(x, w, bias=b)
        got = ops.gemm_f32_few(x, w, b)
        if same_order(m, 2 * n, k):
            assert torch.equal(got, ops.swiglu(both))
        gate, up = both.double().chunk(2, -1)
        want = gate * torch.sigmoid(gate) * up
        # a sum of K terms that add up to some 2 sqrt(K) in magnitude, in either order, and four roundings behind it
        error = (k + 8) * 2.0 ** -24 * 2 * 3 * (1 + gate.abs()) * (1 + up.abs())
        assert bool(((got - want).abs() <= error).all())


@pytest.mark.parametrize("m", [1, 8, 9, 16])
@pytest.mark.parametrize("heads", [(1, 1, 16), (4, 2, 64), (3, 3, 80), (32, 8, 64)])
@pytest.mark.parametrize("turned", [True, False])
@pytest.mark.parametrize("k", [320, 36])
def test_rotation_and_append(m, heads, turned, k):
    nq, nkv, d = heads
    page, pages = 16, 3 * m + 2
    n = (nq + 2 * nkv) * d
    x, w, bias = draw(m + d, (m, k), (n, k), (n,))
    gen = torch.Generator().manual_seed(m)
    positions = torch.randint(0, 3 * page, (m,), generator=gen).int().cuda()
    table = torch.randperm(pages, generator=gen)[: 3 * m].view(m, 3).int().cuda()
    req = torch.randperm(m, generator=gen).int().cuda()
    angles = torch.rand((3 * page, d // 2), generator=torch.Generator(device="cuda").manual_seed(1), device="cuda") * 6
    cos, sin = (angles.cos().contiguous(), angles.sin().contiguous()) if turned else (None, None)

    def caches():
        return (torch.full(ops.key_pages_shape(pages, nkv, page, d), 7.0, device="cuda"),
                torch.full(ops.value_pages_shape(pages, nkv, page, d), 7.0, device="cuda"))

    plain = ops.gemm_generic(x, w, bias=bias)
    want_k, want_v = caches()
    ops.rope_append(plain, positions, req, table, cos, sin, want_k, want_v, nq, nkv, d, page)
    keys, values = caches()
    q = ops.gemm_f32_few(x, w, bias, RopeAppend(positions, req, table, cos, sin, keys, values, nq, nkv, d, page))
    assert q.shape == (m, nq * d)
    for got, want in ((q, plain[:, : nq * d]), (keys, want_k), (values, want_v)):
        if same_order(m, n, k):
            assert torch.equal(got, want)
        else:  # sums of K terms of about one each, in two orders, turned
            assert float((got - want).abs().max()) <= 2 * (k + 4) * 2.0 ** -24 * k


def test_what_is_refused():
    x, w = draw(0, (4, 64), (96, 64))
    for bad_x, bad_w in ((torch.randn(17, 64, device="cuda"), w), (x[:, 1:], w[:, 1:].contiguous()), (x.bfloat16(), w.bfloat16()), (x, w[:95]), (x, w.t())):
        with pytest.raises(KernelError):
            ops.gemm_f32_few(bad_x, bad_w)
