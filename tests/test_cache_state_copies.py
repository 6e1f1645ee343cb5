"""What a step's slots held in the state comes back when the step fails, in whichever order the step names them; other slots are left alone."""

import pytest
import torch

from beholdd.cache.sequence_cache import SequenceCache
from beholdd.parts.base import CacheNeed


@pytest.mark.parametrize("picked", [[0, 1, 2], [1, 2, 3, 4], [3], [2, 1, 0], [0, 2, 4], [4, 0, 1], [1, 2, 4]])
def test_rollback_restores_state_of_any_slots(picked):
    needs = {0: CacheNeed(kind="state", state_shape=(3, 5)), 1: CacheNeed(kind="state", state_shape=(3, 5)), 2: CacheNeed(kind="state", state_shape=(7,))}
    cache = SequenceCache(needs, 640, torch.float32, "cpu", 64, max_slots=6)
    cache.allocate()
    slots = [cache.alloc_slot() for _ in range(6)]
    states = [g.state for g in cache.groups]
    for state in states:
        state.copy_(torch.arange(state.numel(), dtype=torch.float32).view(state.shape))
    before = [state.clone() for state in states]
    requests = [(slots[i], 2) for i in picked]
    cache.reserve(requests)
    for state in states:
        state += 1.0          # every slot: the step's own come back, the others keep what they were given meanwhile
    cache.rollback(requests)
    for state, was in zip(states, before):
        for slot in slots:
            assert torch.equal(state[:, slot], was[:, slot] + (0.0 if slot in [slots[i] for i in picked] else 1.0))
