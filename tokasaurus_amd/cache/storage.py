"""Device tensors behind the cache manager's page ids and slots.

Per group: keys ``[entries, pages, nkv, d / 8, P, 8]`` and values
``[entries, pages, nkv, P / 4, d, 4]``: inside a page the keys lie in pieces of 8
elements and the values in groups of 4 tokens, the order in which the lanes of the
attention kernel read them (``kernels.ops.key_pages_shape``).  The reference keeps
``[pages, P, nkv, d]`` per layer for both (tokasaurus/model/kv_cache.py:27-54).  Per run entry with fixed-size state:
``[slots + 1, *shape]``.  The last page of every pool and the last slot belong to
no request: rows that only pad a step to a recorded size write there (the
reference's scratch page, tokasaurus/model/utils.py:363-369,552-554).
"""

from __future__ import annotations

import torch

from tokasaurus_amd.cache.manager import CacheGroup
from tokasaurus_amd.kernels.ops import key_pages_shape, value_pages_shape
from tokasaurus_amd.parts.base import StateNeed


class CacheStorage:
    def __init__(
        self,
        groups: list[CacheGroup],
        num_pages: list[int],
        page_size: int,
        state_needs: list,  # per run entry: None, a StateNeed, or a list of them
        max_slots: int,
        dtype: torch.dtype,
        device: torch.device,
        embedding_state_need: StateNeed | None = None,
    ):
        self.page_size = page_size
        self.keys: list[torch.Tensor] = []
        self.values: list[torch.Tensor] = []
        for grp, n in zip(groups, num_pages):
            nkv, d = grp.need.num_kv_heads, grp.need.head_dim
            # one page more than the pool hands out: the null page, where padding rows write
            entries = (len(grp.entries),)
            self.keys.append(torch.zeros(entries + key_pages_shape(n + 1, nkv, page_size, d, padded=True), dtype=dtype, device=device))
            self.values.append(torch.zeros(entries + value_pages_shape(n + 1, nkv, page_size, grp.need.value_size), dtype=dtype, device=device))
        def make(need):
            if need is None:
                return None
            if isinstance(need, (list, tuple)):  # a block with several states gets them as a list
                return [make(n) for n in need]
            return torch.zeros((max_slots + 1, *need.shape), dtype=need.dtype, device=device)

        self.states: list = [make(need) for need in state_needs]
        # what the embedding keeps per request (the token before, for one that reads pairs of tokens)
        self.embedding_state = make(embedding_state_need)
        # slot `max_slots` belongs to no request (padding rows of a recorded step use it)
        self.last_token = torch.zeros((max_slots + 1,), dtype=torch.int32, device=device)

    def reset_slots(self, slots: list[int]) -> None:
        """Zero the state of these slots in every state tensor: a request that takes a slot
        starts from the state a fresh engine would give it, whoever held the slot before."""
        if not slots:
            return
        rows: dict[torch.dtype, list[torch.Tensor]] = {}
        for item in [*self.states, self.embedding_state]:
            for t in (item if isinstance(item, list) else [item]):
                if t is not None:
                    rows.setdefault(t.dtype, []).extend(t[s] for s in slots)
        for same in rows.values():
            # one launch for many rows: two requests over six layers of 1.1 MB a row 5.2 us on the device and 19 on the host, row by row 54 and 53
            torch._foreach_zero_(same)

    def bytes(self) -> int:
        return sum(t.numel() * t.element_size() for t in self.keys + self.values)
