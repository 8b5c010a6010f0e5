"""The experts' products in tiles: sizes that end inside a step of K, inside a block of outputs and inside a tile, experts with
no, one and many tiles, empty places, identity experts, weights on either side, against 64-bit sums."""

import pytest
import torch

from tokasaurus_amd.kernels import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens", [13, 129, 700])
@pytest.mark.parametrize("experts,top", [(5, 5), (40, 3), (2, 2)])
@pytest.mark.parametrize("width,ff", [(64, 32), (72, 40), (136, 200), (512, 264)])
@pytest.mark.parametrize("form", ["silu", "clamps", "on input"])
def test_experts_in_tiles(tokens, experts, top, width, ff, form):
    if tokens * top < ops.EXPERT_TILES_FROM_PAIRS:
        tokens = -(-ops.EXPERT_TILES_FROM_PAIRS // top)
    assert ops.experts_go_in_tiles(tokens, top, torch.bfloat16, width, ff)
    g = torch.Generator(device="cuda").manual_seed(tokens + experts + width)
    rand = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    h = rand(tokens, width + 8).bfloat16()[:, :width]  # rows a stride apart
    gu, dn = (rand(experts, 2 * ff, width) * width ** -0.5).bfloat16(), (rand(experts, width, ff) * ff ** -0.5).bfloat16()
    skew = torch.rand((tokens, experts + 2), generator=g, device="cuda") ** torch.linspace(1, 4, experts + 2, device="cuda")
    ids = skew.argsort(-1, descending=True)[:, :top].to(torch.int32).contiguous()  # some experts have many tokens; two are identities
    ids[::7, 0] = -1
    if form == "on input":
        ids[ids >= experts] = -1
    weights = torch.rand((tokens, top), generator=g, device="cuda")
    limit, alpha = (1.5, 1.702) if form == "clamps" else (0.0, 0.0)
    got = ops.expert_mix(h, gu, dn, ids, weights, weights_on_input=form == "on input", glu=(limit, alpha) if limit else None)
    hd, want = h.double(), torch.zeros((tokens, width), dtype=torch.float64, device="cuda")
    for e in range(experts + 2):
        for k in range(top):
            rows = (ids[:, k] == e).nonzero()[:, 0]
            w = weights[rows, k : k + 1].double()
            if e >= experts:
                want[rows] += w * hd[rows]
                continue
            y = hd[rows] @ gu[e].double().T
            y = y * w if form == "on input" else y
            a, u = y[:, :ff], y[:, ff:]
            if limit:
                a, u = a.clamp(max=limit), u.clamp(-limit, limit)
                z = a * torch.sigmoid(alpha * a) * (u + 1)
            else:
                z = a * torch.sigmoid(a) * u
            y = z @ dn[e].double().T
            want[rows] += y if form == "on input" else w * y
    # roundings to bfloat16, each at most 2^-9 of a value: gate, up, the activation, their product, the expert's row; a row's
    # error is then within 5 * 2^-9 of its terms, and these add like independent ones
    assert float((got.double() - want).norm() / want.norm()) <= 5 * 2.0 ** -9
    assert torch.isfinite(got).all()
