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


@pytest.mark.parametrize("tokens", [40, 257, 700])
@pytest.mark.parametrize("experts,top", [(5, 3), (2, 2), (1, 1)])
@pytest.mark.parametrize("width,ff", [(64, 64), (320, 192), (512, 1088)])
@pytest.mark.parametrize("form", ["silu", "clamps", "on input"])
def test_experts_in_pairs_of_tiles(monkeypatch, tokens, experts, top, width, ff, form):
    """One step of K, fewer than local memory holds, and more; outputs that end inside a block; no, one and several pairs."""
    for least in ("ROWS", "WIDTH", "INNER", "WALK"):
        monkeypatch.setattr(ops, f"EXPERT_PAIRS_FROM_{least}", 0)
    assert ops.experts_go_in_pairs_of_tiles(tokens * top, experts, width + 8, width, ff)
    test_experts_in_tiles(tokens, experts, top, width, ff, form)


@pytest.mark.parametrize("pairs,experts,width,ff,wanted", [
    (16384, 32, 2048, 1024, True), (15000, 32, 2048, 1024, False), (8000, 16, 2048, 2048, True), (6700, 16, 2048, 2048, False), (51200, 128, 2048, 768, True),
    (38400, 128, 2048, 768, False), (67840, 64, 1024, 512, False), (3040, 8, 4096, 14336, True), (3680, 8, 4096, 1792, False), (5280, 8, 4096, 1792, True),
    (51200, 128, 2048, 760, False), (51200, 128, 2056, 768, False)])
def test_which_experts_go_in_pairs_of_tiles(pairs, experts, width, ff, wanted):
    assert ops.experts_go_in_pairs_of_tiles(pairs, experts, width, width, ff) == wanted


@pytest.mark.parametrize("tokens,top,experts", [(1, 1, 300), (13, 8, 256), (130, 1, 2), (129, 1, 1), (400, 3, 5), (64, 2, 64)])
@pytest.mark.parametrize("spread", ["one expert", "all", "each its own"])
def test_tiles_hold_every_choice(tokens, top, experts, spread):
    """The fewest tiles that can hold any choice: all pairs on one expert, on all alike, and a pair an expert as far as they go."""
    pairs = tokens * top
    if spread == "one expert":
        ids = torch.full((tokens, top), experts - 1, dtype=torch.int32)
    elif spread == "all":
        ids = (torch.arange(pairs, dtype=torch.int32) % experts).view(tokens, top)
    else:  # every expert but one has one pair, the last all others
        ids = torch.arange(pairs, dtype=torch.int32).clamp(max=min(experts, pairs) - 1).view(tokens, top)
    s = ops.expert_sort([(ids.cuda(), experts)])[0]
    assert s.max_tiles == ops.expert_tiles(pairs, experts) <= pairs
    used = int(s.tile_group[-1])
    count = torch.bincount(ids.flatten().long(), minlength=experts)
    assert used == int((-(-count // ops.EXPERT_TILE)).sum()) <= s.max_tiles
    slot_pair, group = s.slot_pair.cpu().view(-1, ops.EXPERT_TILE), s.tile_group.cpu()
    assert sorted(slot_pair[slot_pair >= 0].tolist()) == list(range(pairs))
    runs = s.runs.cpu().view(-1, 4).tolist()  # every used tile in one pair of its expert, the last one perhaps alone in it
    mine = [(t + 2 * (i - first) + j, e) for i, (t, e, first, tiles) in enumerate(runs[1 : 1 + runs[0][0]]) for j in range(2) if 2 * (i - first) + j < tiles]
    assert mine == list(enumerate(group[:used].tolist())) and runs[0][0] <= s.max_pairs
    for t in range(s.max_tiles):
        mine = slot_pair[t][slot_pair[t] >= 0].long()
        assert (t < used) == (mine.numel() > 0) and (ids.flatten()[mine] == group[t]).all()


@pytest.mark.parametrize("spread", ["one expert", "all", "each its own"])
def test_as_many_experts_as_local_memory_holds(spread):
    """4,096 experts, three numbers each: 48 KB, which a kernel has without asking for more; one expert more is refused."""
    test_tiles_hold_every_choice(700, 8, 4096, spread)
    with pytest.raises(ops.KernelError, match="too many experts"):
        ops.expert_sort([(torch.zeros((2, 2), dtype=torch.int32, device="cuda"), 4097)])


def test_room_for_the_experts_is_that_of_the_pairs():
    """256 experts of inner size 2,048, 64 pairs: rows between the two products are the pairs', not those of tiles an expert."""
    g = torch.Generator(device="cuda").manual_seed(1)
    h = torch.randn((32, 64), generator=g, device="cuda").bfloat16()
    gu = torch.randn((256, 4096, 64), generator=g, device="cuda").bfloat16()
    dn = torch.randn((256, 64, 2048), generator=g, device="cuda").bfloat16()
    ids, weights = torch.randint(0, 256, (32, 2), generator=g, device="cuda", dtype=torch.int32), torch.rand((32, 2), generator=g, device="cuda")
    pairs = ops.expert_sort([(ids, 256)])[0]
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    out = ops.expert_mix(h, gu, dn, ids, weights, pairs=pairs)
    assert torch.isfinite(out).all() and torch.cuda.max_memory_allocated() - before < 4 << 20


@pytest.mark.parametrize("tokens,experts,top,width,ff", [(257, 3, 2, 64, 4224), (700, 90, 3, 1600, 64), (385, 1, 1, 320, 192), (320, 1, 1, 192, 320),
                                                         (321, 1, 1, 64, 64), (65, 1, 1, 64, 128), (900, 40, 3, 320, 192)])
@pytest.mark.parametrize("form", ["silu", "on input"])
def test_odd_tiles_apart_and_beside_their_pairs(monkeypatch, tokens, experts, top, width, ff, form):
    """An inner size beyond which odd tiles stay beside their pairs, experts enough that they do, and odd tiles of 1, 64 and 65 rows and of
    more apart."""
    test_experts_in_pairs_of_tiles(monkeypatch, tokens, experts, top, width, ff, form)


@pytest.mark.parametrize("tokens,top,experts", [(130, 1, 2), (400, 3, 5), (64, 2, 64), (1000, 4, 3)])
def test_whole_pairs_and_odd_tiles_are_listed_apart(tokens, top, experts):
    """Every tile that is used once, in a whole pair or as an odd one with the rows that it holds."""
    ids = torch.randint(0, experts, (tokens, top), dtype=torch.int32, generator=torch.Generator().manual_seed(tokens))
    s = ops.expert_sort([(ids.cuda(), experts)])[0]
    runs, group = s.runs.cpu().view(-1, 4).tolist(), s.tile_group.cpu().tolist()
    pairs, whole, odd, _ = runs[0]
    order = runs[1 + s.max_pairs : 1 + 2 * s.max_pairs]
    assert pairs == whole + odd
    tiles = []
    for i, (tile, e, first, count) in enumerate(order[:whole]):
        assert first <= i < first + count
        tiles += [(tile + 2 * (i - first) + j, e) for j in range(2)]
    counts = torch.bincount(ids.flatten().long(), minlength=experts).tolist()
    for tile, e, rows, _ in order[len(order) - odd :]:
        assert rows == (counts[e] - 1) % ops.EXPERT_TILE + 1
        tiles.append((tile, e))
    assert sorted(tiles) == list(enumerate(group[: group[-1]]))


def test_room_that_is_no_list_of_the_tiles_pairs_is_refused(monkeypatch):
    """The grid of the pairs comes from how many tiles and pairs there can be: fewer pairs than half the tiles would leave tiles out."""
    import dataclasses

    for least in ("ROWS", "WIDTH", "INNER", "WALK"):
        monkeypatch.setattr(ops, f"EXPERT_PAIRS_FROM_{least}", 0)
    g = torch.Generator(device="cuda").manual_seed(1)
    tokens, experts, width, ff = 771, 3, 64, 64
    h = torch.randn((tokens, width), generator=g, device="cuda").bfloat16()
    gu, dn = (torch.randn(s, generator=g, device="cuda").bfloat16() for s in ((experts, 2 * ff, width), (experts, width, ff)))
    ids = (torch.arange(tokens, dtype=torch.int32) % experts).view(tokens, 1).cuda()  # 257 rows an expert: a whole pair and an odd tile each
    pairs = ops.expert_sort([(ids, experts)])[0]
    assert pairs.max_tiles == 9 and pairs.runs[:3].tolist() == [6, 3, 3]
    got = ops.expert_mix(h, gu, dn, ids, None, pairs=pairs)
    for e in range(experts):
        y = h[e::experts].double() @ gu[e].double().T
        act = (torch.nn.functional.silu(y[:, :ff]) * y[:, ff:]).bfloat16().double()
        want, size = act @ dn[e].double().T, act.abs() @ dn[e].double().abs().T
        # gate, up, silu and their product are rounded to 8 bits in front of the sums, a row behind them
        assert ((got[e::experts].double() - want).abs() <= 2.0 ** -6 * (size + want.abs())).all()
    with pytest.raises(ops.KernelError, match="pairs of 9 tiles"):
        ops.expert_mix(h, gu, dn, ids, None, pairs=dataclasses.replace(pairs, max_pairs=4))


@pytest.mark.parametrize("counts", [[0, 1, 64, 65, 128, 129, 256, 257, 320, 321], [640, 192, 448, 511], [64] * 70])
def test_odd_tiles_of_few_rows_are_counted(counts):
    """Experts whose odd last tile has up to 64 rows, beside whole pairs and odd tiles."""
    ids = torch.cat([torch.full((n,), e, dtype=torch.int32) for e, n in enumerate(counts)])
    s = ops.expert_sort([(ids[torch.randperm(len(ids), generator=torch.Generator().manual_seed(1))].view(-1, 1).cuda(), len(counts))])[0]
    tiles = [-(-n // 128) for n in counts]
    assert s.runs[:4].tolist() == [sum((t + 1) // 2 for t in tiles), sum(t // 2 for t in tiles), sum(t % 2 for t in tiles),
                                   sum(t % 2 == 1 and n - 128 * (t - 1) <= 64 for n, t in zip(counts, tiles))]


@pytest.mark.parametrize("counts", [[520, 640, 300, 129], [270] * 4, [512, 768, 256, 1024]])
def test_odd_tiles_apart_and_beside(counts, monkeypatch):
    """Where odd tiles behind the pairs save a round (many outputs) and where they do not, or there are none: the same bits, those of tiles by themselves."""
    for least in ("ROWS", "WIDTH", "INNER", "WALK"):
        monkeypatch.setattr(ops, f"EXPERT_PAIRS_FROM_{least}", 0)
    g = torch.Generator(device="cuda").manual_seed(1)
    ids = torch.cat([torch.full((n,), e, dtype=torch.int32) for e, n in enumerate(counts)]).view(-1, 1).cuda()
    for width, ff in ((64, 64), (128, 12288)):  # (96 blocks of gate and up: several rounds of workgroups)
        h = torch.randn((len(ids), width), generator=g, device="cuda").bfloat16()
        gu, dn = ((torch.randn(s, generator=g, device="cuda") * 0.1).bfloat16() for s in ((len(counts), 2 * ff, width), (len(counts), width, ff)))
        got = ops.expert_mix(h, gu, dn, ids, None)
        monkeypatch.setattr(ops, "experts_go_in_pairs_of_tiles", lambda *a: False)
        want = ops.expert_mix(h, gu, dn, ids, None)
        monkeypatch.undo()
        for least in ("ROWS", "WIDTH", "INNER", "WALK"):
            monkeypatch.setattr(ops, f"EXPERT_PAIRS_FROM_{least}", 0)
        # the activations' 8 bits (off by one rounding where the orders of 32-bit sums differ) and the sums behind them
        assert float((got.double() - want.double()).norm()) <= 2.0 ** -7 * float(want.double().norm())
