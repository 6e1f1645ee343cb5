"""Captures of decode steps: when the one before is dropped, and where device memory runs short."""

import pytest
import torch

pytestmark = pytest.mark.gpu

CONFIG = {"architectures": ["Qwen3ForCausalLM"], "num_hidden_layers": 2, "hidden_size": 64, "num_attention_heads": 4, "num_key_value_heads": 2, "head_dim": 32,
          "intermediate_size": 96, "vocab_size": 200, "rope_theta": 1000000.0, "rms_norm_eps": 1e-6, "max_position_embeddings": 512, "tie_word_embeddings": False}


def steps(folder, counts, held=None, **options):
    """The logits of decode steps of so many sequences each, of three that have had a prompt."""
    import beholdd
    engine = beholdd.Engine(folder, dtype="bfloat16", max_tokens=1024, max_slots=3, device="cuda:0", **options)
    slots = [engine.alloc_slot() for _ in range(3)]
    engine.step([beholdd.StepEntry(slot, [7, slot + 1, 3], []) for slot in slots])
    out = []
    for at, count in enumerate(counts):
        logits = engine.step([beholdd.StepEntry(slot, [at + 5], [0]) for slot in slots[:count]])
        if held is not None:
            held.append(logits)      # what a capture that is dropped has returned
        out.append(logits.clone())
    return out


@pytest.fixture()
def folder(tmp_path):
    import beholdd
    return beholdd.write_random_model(str(tmp_path), CONFIG, seed=2, dtype="bfloat16", std=0.05)


@pytest.mark.parametrize("limit", [0, 1, 2])
def test_a_capture_after_the_last_one_was_dropped(folder, limit):
    counts = [2, 3, 3, 2, 2, 1, 2, 3, 3]
    want = steps(folder, counts)      # all of them kept
    for held in (None, []):
        got = steps(folder, counts, held, graph_limit=limit)
        assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("short", [False, True])
def test_cached_memory_is_given_back_before_a_capture_that_might_need_it(folder, monkeypatch, short):
    real, total = torch.cuda.mem_get_info, torch.cuda.get_device_properties(0).total_memory
    given_back = []
    # free: what is cached and no more, which leaves nothing for the logits and for segments that the pool opens
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda device=None: (torch.cuda.memory_reserved() - torch.cuda.memory_allocated() + 512, total) if short else real(device))
    monkeypatch.setattr(torch.cuda, "empty_cache", lambda: given_back.append(1))
    steps(folder, [3, 3, 2, 3])
    assert len(given_back) == (2 if short else 0)


def test_a_process_that_may_have_a_part_of_the_memory_only_gives_back_as_well(folder, monkeypatch):
    given_back = []
    monkeypatch.setattr(torch.cuda, "get_per_process_memory_fraction", lambda device=None: torch.cuda.memory_reserved() / torch.cuda.get_device_properties(0).total_memory)
    monkeypatch.setattr(torch.cuda, "empty_cache", lambda: given_back.append(1))
    steps(folder, [3, 3])
    assert len(given_back) == 1
