"""The state of requests that take a slot starts at zero, in every state tensor, and nobody else's does."""

import pytest
import torch

from tokasaurus_amd.cache.storage import CacheStorage
from tokasaurus_amd.parts.base import StateNeed


@pytest.mark.parametrize("slots", [[], [0], [4, 1], [0, 1, 2, 3, 4]])
@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_only_these_slots(slots, device):
    needs = [None, StateNeed((3, 5)), [StateNeed((7,), torch.bfloat16), StateNeed((2, 2, 3))], StateNeed((1,), torch.int32)]
    storage = CacheStorage([], [], 16, needs, 5, torch.bfloat16, torch.device(device), StateNeed((2,), torch.int32))
    states = [storage.states[1], *storage.states[2], storage.states[3], storage.embedding_state]
    for t in states:
        t.fill_(3)
    storage.reset_slots(slots)
    for t in states:
        for s in range(6):
            assert bool((t[s] == (0 if s in slots else 3)).all())
