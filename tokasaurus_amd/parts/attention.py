"""Grouped-query attention over the paged cache
(tokasaurus/model/llama.py:96-287, tokasaurus/model/attention_utils.py:87-175).

q, k and v are one stacked product; the rotation of q and k is fused with the
append of k and v to the request's pages; one attention call then serves
prompt portions and single decoded tokens alike, each token reading the keys
at positions up to its own (bottom-right aligned causal mask), optionally only
the last ``window`` of them.
"""

from __future__ import annotations

import math
from dataclasses import dataclass

import torch

from tokasaurus_amd.kernels import ops
from tokasaurus_amd.kernels.upload import upload
from tokasaurus_amd.parts.base import (
    NORM_WEIGHT,
    MIXERS,
    POSITION_ENCODINGS,
    CacheNeed,
    CacheView,
    Mixer,
    Normed,
    PartSpec,
    StepContext,
    TensorSpec,
)
from tokasaurus_amd.parts.grouped_attention import tile_plan
from tokasaurus_amd.parts.linear import Linear, Placer


@dataclass
class AttentionLaunch:
    """One call of the matrix-core kernel: the tiles of some of the step's requests."""

    tile_req: torch.Tensor
    tile_row0: torch.Tensor
    tile_row1: torch.Tensor | None
    row_tiles: int
    split: int
    waves: int
    max_kv_len: int  # bounds the keys of the launch's requests: sizes its grid and scratch
    scratch: ops.AttentionScratch | None = None  # a replayed step keeps its own
    grouped: int = 0  # 1, 2: tiles in groups of one request that share their loads, with so many sets of wavefronts (long prompts)
    even: bool = False  # decoded tokens: the wavefronts of a workgroup share the keys that are there, not the split


@dataclass
class AttentionPlan:
    """How the step's rows are cut into tiles and its keys into splits; made once
    a step for each group size and shared by the layers.  Requests that bring one
    row tile or less (decoded tokens) get wavefronts of one row tile and split keys;
    prompt portions get wavefronts of two row tiles and whole keys: an early tile paired with
    a late one, or single or neighbouring tiles whose keys two wavefronts share (``ops.attention_prompt_form``),
    or, when there are enough of them and a page holds 16 keys or more, neighbouring
    tiles in groups of four wavefronts that share every load of keys and values (with two such
    sets of wavefronts a group while the groups are too few to fill the chip several times
    over: ``ops.attention_group_sets``); portions that fill few wavefronts but walk many keys
    (a short portion after a long past) get their keys cut like decoded tokens' and a second
    kernel that adds the splits (``ops.attention_prompt_split``)."""

    launches: list[AttentionLaunch]
    max_kv_len: int


def attention_plan(ctx: StepContext, group: int, nkv: int, head_dim: int, page_size: int) -> AttentionPlan:
    key = ("attention_plan", group, nkv, head_dim, page_size)
    plan = ctx.extras.get(key)
    if plan is None:
        q_lens = [ctx.host_q_start[i + 1] - ctx.host_q_start[i] for i in range(ctx.num_requests)]
        small = [r for r, n in enumerate(q_lens) if 0 < n * group <= 16]
        large = [r for r, n in enumerate(q_lens) if n * group > 16]
        static = bool(ctx.extras.get("static"))
        # launches are chosen for the bound the step was planned for, not for the lengths in it (but for decoded rows beside prompts,
        # which no recorded step holds: they are cut by their own lengths)
        bound = max(int(ctx.extras.get("kv_bound", 0)), ctx.max_kv_len)
        lists: list[tuple[list[int], list[int], list[int] | None, int, int, int, int, int, bool]] = []
        if small:
            req, row0, _ = ops.attention_tiles(q_lens, group, 1, small)
            if large and not static:
                lengths = [ctx.host_kv_len[r] for r in small]
                split, waves = ops.attention_even_split(lengths, nkv, head_dim, group)
                even = (split, waves) != ops.attention_split(max(lengths), len(req), nkv, head_dim, group)
                lists.append((req, row0, None, 1, split, waves, 0, max(lengths), even))
            else:
                split, waves = ops.attention_split(bound, len(req), nkv, head_dim, group)
                even = ops.attention_even_parts(bound, len(req), nkv, head_dim, waves)
                lists.append((req, row0, None, 1, split, waves, 0, bound, even))
        # Portions that come after a past several times their own length walk far more keys a row than
        # whole prompts do: they are planned apart, or one of them among whole prompts would take a
        # form chosen for the many short walks and walk its long past on a few wavefronts.
        # (and among them the short ones, whose keys are cut, apart from the long ones, which fill the chip as they are)
        own = lambda r: -(-q_lens[r] * group // 32) * nkv  # the request's wavefronts of two row tiles
        long_past = lambda r: ctx.host_kv_len[r] >= 2048 and ctx.host_kv_len[r] >= 4 * q_lens[r]
        fresh = [r for r in large if not long_past(r)]
        tails = [r for r in large if long_past(r) and own(r) <= 512]
        after_past = [r for r in large if long_past(r) and own(r) > 512]
        whole = -(-max(bound, 1) // 128) * 128

        def longest_first(req: list[int], row0: list[int], unit: int) -> tuple[list[int], list[int]]:
            """The tiles by the keys they walk, ``unit`` of them together: what starts last is short, of whichever request.  us a layer, 8 kv
            heads, request by request / so: 4 x 1,024 tokens of 32 heads of 128 74.3 / 61.0, of 64 53.1 / 45.9, 2 x 2,048 of 64 75.9 / 67.7."""
            reach = lambda i: max(ctx.host_kv_len[req[j]] - q_lens[req[j]] + row0[j] // group for j in range(i, i + unit))  # noqa: E731
            order = [j for i in sorted(range(0, len(req), unit), key=reach, reverse=True) for j in range(i, i + unit)]
            return [req[j] for j in order], [row0[j] for j in order]

        for some in (fresh, after_past, tails):
            if not some:
                continue
            wavefronts = sum(-(-q_lens[r] * group // 32) for r in some) * nkv
            longest = max(ctx.host_kv_len[r] for r in some)
            split = ops.attention_prompt_split(wavefronts, head_dim, longest)
            sets = 0 if split else ops.attention_group_sets(wavefronts, head_dim, page_size, longest)
            if sets:
                req, row0, _ = ops.attention_tiles(q_lens, group, 2, some, fill=ops.ATTENTION_GROUP)
                req, row0 = longest_first(req, row0, ops.ATTENTION_GROUP)
                lists.append((req, row0, None, 2, whole, 1, sets, bound, False))
                continue
            row_tiles, waves = (2, 1) if split else ops.attention_prompt_form(wavefronts, head_dim, longest)
            if waves > 1:
                req, row0, _ = ops.attention_tiles(q_lens, group, row_tiles, some)
                req, row0 = longest_first(req, row0, 1)
                lists.append((req, row0, None, row_tiles, whole, waves, 0, bound, True))
            else:
                # (cut keys: the grid and the scratch are sized for these requests, not for a longer one that decodes beside them)
                req, row0, row1 = ops.attention_tiles(q_lens, group, 2, some, pair=True)
                lists.append((req, row0, row1, 2, split or whole, 1, 0, longest if split else bound, False))
        # one upload for all the tile lists of the step
        flat = [x for req, row0, row1, *_ in lists for x in (req + row0 + (row1 or []))]
        dev = upload(flat, torch.int32, ctx.device) if flat else None
        launches, at = [], 0
        for req, row0, row1, row_tiles, split, waves, grouped, max_kv_len, even in lists:
            n = len(req)
            t_req, t_row0 = dev[at : at + n], dev[at + n : at + 2 * n]
            t_row1 = dev[at + 2 * n : at + 3 * n] if row1 is not None else None
            at += (3 if row1 is not None else 2) * n
            launches.append(AttentionLaunch(t_req, t_row0, t_row1, row_tiles, split, waves, max_kv_len,
                                            ops.AttentionScratch(ctx.device) if static else None, grouped, even))
        plan = AttentionPlan(launches, bound)
        ctx.extras[key] = plan
    return plan


@MIXERS.register("paged_attention")
class PagedAttention(Mixer):
    fuses_norm = True

    def __init__(
        self,
        hidden_size: int,
        num_heads: int,
        num_kv_heads: int,
        head_dim: int,
        names: dict[str, str],
        position: PartSpec | None = None,
        window: int = 0,
        shared: dict | None = None,
        bias_names: dict[str, str] | None = None,
        rotary_dim: int | None = None,
        head_norm: dict | None = None,
    ):
        """``names``: checkpoint names of the q, k, v and o matrices; ``bias_names``: of the bias
        vectors of those among them that have one (keys "q", "k", "v", "o").  ``rotary_dim``: the
        leading elements of every head that the position encoding rotates (the whole head when
        None); the encoding's tables must then have rotary_dim / 2 entries a position.
        ``head_norm``: ``{"q": name, "k": name, "eps": eps}``: every query head and every key head
        passes an RMSNorm over its own elements (one weight [head_dim] for the queries, one for the
        keys) between the projection and the rotation."""
        if num_heads % num_kv_heads:
            raise ValueError(f"{num_heads} query heads are not a multiple of {num_kv_heads} kv heads")
        if rotary_dim is not None and not (0 < rotary_dim <= head_dim and rotary_dim % 2 == 0):
            raise ValueError(f"rotary_dim {rotary_dim} must be even and at most the head size {head_dim}")
        self.rotary_dim = None if rotary_dim in (None, head_dim) else int(rotary_dim)
        self.head_norm = dict(head_norm) if head_norm else None
        self.q_norm_weight: torch.Tensor | None = None
        self.k_norm_weight: torch.Tensor | None = None
        bias_names = bias_names or {}
        self.hidden_size = hidden_size
        self.num_heads = num_heads
        self.num_kv_heads = num_kv_heads
        self.head_dim = head_dim
        self.window = int(window)
        self.scale = 1.0 / math.sqrt(head_dim)
        self.qkv = Linear(
            hidden_size,
            [names["q"], names["k"], names["v"]],
            [num_heads * head_dim, num_kv_heads * head_dim, num_kv_heads * head_dim],
            [bias_names.get("q"), bias_names.get("k"), bias_names.get("v")],
        )
        self.out = Linear(num_heads * head_dim, [names["o"]], [hidden_size], [bias_names.get("o")])
        self.position = None
        if position is not None:
            shared = shared if shared is not None else {}
            self.position = shared.setdefault(("position", position), POSITION_ENCODINGS.build(position))

    def tensor_specs(self) -> list[TensorSpec]:
        specs = self.qkv.tensor_specs() + self.out.tensor_specs()
        if self.head_norm:
            specs += [TensorSpec(self.head_norm[x], (self.head_dim,), NORM_WEIGHT) for x in ("q", "k")]
        return specs

    def cache_need(self) -> CacheNeed:
        return CacheNeed(self.num_kv_heads, self.head_dim, self.window)

    def check_cache(self, page_size: int, dtype: torch.dtype) -> None:
        ops.check_attention_shape(dtype, self.num_heads, self.num_kv_heads, self.head_dim, page_size)

    def load(self, tensors: dict[str, torch.Tensor], placer: Placer) -> None:
        self.qkv.load(tensors, placer)
        self.out.load(tensors, placer)
        if self.head_norm:
            def place(name: str) -> torch.Tensor:
                host = tensors[name]
                dtype = torch.float32 if host.dtype == torch.float32 else placer.dtype
                return placer.place(("vector", name), lambda: host.to(dtype=dtype).contiguous().to(placer.device))

            self.q_norm_weight, self.k_norm_weight = place(self.head_norm["q"]), place(self.head_norm["k"])
        if self.position is not None:
            self.position.prepare(placer.device)

    def forward(
        self,
        h: torch.Tensor | Normed,
        residual: torch.Tensor,
        ctx: StepContext,
        cache: CacheView | None,
        state: torch.Tensor | None,
        rows: torch.Tensor | None,
        emit_norm=None,
    ):
        assert cache is not None, "paged attention needs a cache"
        nq, nkv, d = self.num_heads, self.num_kv_heads, self.head_dim
        cos = self.position.cos if self.position is not None else None
        sin = self.position.sin if self.position is not None else None
        q = None
        if cache.writable and not self.head_norm:
            # few rows in bfloat16: one kernel multiplies, rotates and appends
            q = self.qkv.rope_append(h, ops.RopeAppend(
                ctx.positions, ctx.token_req, cache.block_table, cos, sin, cache.keys, cache.values,
                nq, nkv, d, cache.page_size, self.rotary_dim))
        if q is None:
            # an entry that reads another entry's cache computes only its queries
            q = self.qkv(h, rows=None if cache.writable else nq * d)
            if self.head_norm:  # per-head norms stand between the projection and the rotation
                eps = float(self.head_norm["eps"])
                ops.head_rmsnorm(q, self.q_norm_weight, eps, 0, nq, d)
                if cache.writable:
                    ops.head_rmsnorm(q, self.k_norm_weight, eps, nq, nkv, d)
            ops.rope_append(
                q, ctx.positions, ctx.token_req, cache.block_table, cos, sin,
                cache.keys, cache.values, nq, nkv, d, cache.page_size, write_cache=cache.writable,
                rotary_dim=self.rotary_dim,
            )
        if ops.attention_mfma_supports(q.dtype, d, cache.page_size):
            plan = attention_plan(ctx, nq // nkv, nkv, d, cache.page_size)
            attn = torch.empty((q.shape[0], nq * d), dtype=q.dtype, device=q.device)
            for launch in plan.launches:
                ops.paged_attention_mfma(
                    q, cache.keys, cache.values, cache.block_table, ctx.q_start, ctx.kv_len,
                    launch.tile_req, launch.tile_row0, launch.row_tiles, nq, nkv, d, cache.page_size,
                    launch.max_kv_len, launch.split, window=self.window, scale=self.scale, waves=launch.waves,
                    out=attn, scratch=launch.scratch, tile_row1=launch.tile_row1, longest=min(ctx.max_kv_len, launch.max_kv_len),
                    grouped=launch.grouped, even=launch.even,
                )
        elif q.dtype == torch.float32 and ops.attention_tile_f32_fits(nq, nkv, d, d, cache.page_size):
            # the true 32-bit path: 32-bit products on the matrix cores, prompt portions in tiles of 16 tokens, single
            # tokens (which come behind them) in tiles of the heads that share a kv head.  Steps of the 1B shape with the
            # plain kernel here and with this one: one row after 64 tokens 1.7 ms with either, 4 after 6,000 tokens 38 and 2.2
            # ms, 3 of 280 to 2,223 tokens beside two prompts of 33 in all 45 and 3.0 ms
            attn = torch.empty((q.shape[0], nq * d), dtype=q.dtype, device=q.device)
            portions, bound = int(ctx.extras.get("num_portions", 0)), ctx.extras.get("kv_bound", ctx.max_kv_len)
            for first, end, longest_q in ((0, portions, 2), (portions, ctx.num_requests, 1)):
                if first == end:
                    continue
                gg = ops.attention_tile_heads(nq // nkv, longest_q)
                tile_req, tile_row0 = tile_plan(ctx, 16 // gg, first, end)
                ops.attention_tile_f32(
                    q, cache.keys, cache.values, cache.block_table, ctx.q_start, ctx.kv_len, tile_req, tile_row0, nq, nkv, d, d,
                    cache.page_size, gg, window=self.window, scale=self.scale, key_chunk=256, longest=bound, out=attn,
                    step_longest=ctx.max_kv_len)
        else:
            # shapes that neither matrix-core kernel takes
            attn = ops.paged_attention_generic(
                q, cache.keys, cache.values, cache.block_table, ctx.token_req, ctx.positions,
                nq, nkv, d, cache.page_size, window=self.window, scale=self.scale,
            )
        if rows is not None:
            attn = ops.gather_rows(attn, rows)
        return self.out.with_residual(attn, residual, emit_norm)
