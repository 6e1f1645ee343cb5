"""A state in two rows a slot: which row holds it before and after steps that succeed and fail, and which caches keep one."""

import pytest
import torch

from beholdd.cache.sequence_cache import SequenceCache
from beholdd.parts.base import CacheNeed

NEEDS = {0: CacheNeed(kind="state", state_shape=(3, 5), in_banks=True), 1: CacheNeed(kind="kv", kv_heads=2, head_dim=8, state_shape=(7,), in_banks=True),
         2: CacheNeed(kind="state", state_shape=(4,)), 3: CacheNeed(kind="state", state_shape=(3, 5), in_banks=True)}


def made(banks=(0, 1, 2, 3)):
    cache = SequenceCache(NEEDS, 640, torch.float32, "cpu", 64, max_slots=6, banks=banks)
    plan = cache.allocate()
    assert cache.allocated_bytes() == plan.total_bytes
    return cache


def states(cache):
    return {entry: cache.group_of_entry[entry].state[cache.group_of_entry[entry].index_of[entry]] for entry in NEEDS}


def step(cache, slots, value, fails=False):
    """A step whose layers leave `value` times (entry + 1) in their rows."""
    requests = [(slot, 1) for slot in slots]
    cache.reserve(requests)
    read, to = cache.state_rows(slots)
    for entry, state in states(cache).items():
        state[to if cache.layer_cache(entry, True, {1: None}).banked else slots] = value * (entry + 1.0)
    (cache.rollback if fails else cache.commit)(requests)


def held(cache, slot):
    (row,), _ = cache.state_rows([slot])
    return {entry: float(state[row if cache.layer_cache(entry, True, {1: None}).banked else slot].mean()) for entry, state in states(cache).items()}


@pytest.mark.parametrize("banks", [(0, 1, 2, 3), (0, 3), (0,), ()])
def test_a_step_leaves_the_state_in_the_other_row(banks):
    cache = made(banks)
    by_entry = {entry: cache.layer_cache(entry, True, {1: None}).banked for entry in NEEDS}
    assert by_entry == {0: 3 in banks, 1: 1 in banks, 2: False, 3: 3 in banks}      # a group's entries all, or none of them
    for entry, state in states(cache).items():
        assert state.shape[0] == (12 if by_entry[entry] else 6)
    slots = [cache.alloc_slot() for _ in range(6)]
    expected = {slot: 0.0 for slot in slots}
    for value, some, fails in ((1.0, [0, 1, 2], False), (2.0, [2, 0], True), (3.0, [5, 2], False), (4.0, [4], False), (5.0, [2, 1, 0, 5], False), (6.0, slots, True),
                               (7.0, [3, 2, 1], False)):
        step(cache, some, value, fails)
        if not fails:
            expected.update({slot: value for slot in some})
        for slot in slots:
            assert held(cache, slot) == {entry: expected[slot] * (entry + 1) for entry in NEEDS}, (value, slot)
        read, to = cache.state_rows(slots)
        assert sorted(read + to) == list(range(12)) and all({a, b} == {s, s + 6} for s, a, b in zip(slots, read, to))
    cache.free_slot(2)
    assert cache.alloc_slot() == 2 and held(cache, 2) == {entry: 0.0 for entry in NEEDS}      # whichever row its last owner ended in
    cache.check_invariants()


def test_entries_that_two_runs_share_are_moved_on_in_place():
    from beholdd.engine.engine import entries_of_one_run

    class Model:
        schedule = [(0, 0), (1, 1), (0, 2), (1, 1), (2, 3)]

    assert entries_of_one_run(Model()) == {0, 2, 3} and entries_of_one_run(object()) == set()
