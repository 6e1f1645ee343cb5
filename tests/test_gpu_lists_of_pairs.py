"""The lists of the pairs that chose an expert: whole numbers, in order, at the borders of the runs that the waves take."""

import numpy as np
import pytest
import torch

from test_gpu_pudorax import dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    from beholdd.kernels import HipKernels
    return HipKernels("cuda:0")


@pytest.mark.parametrize("rows,top,experts", [(1, 1, 1), (1, 4, 32), (64, 4, 32), (65, 4, 8), (257, 1, 3), (1025, 4, 32), (2100, 4, 32), (5001, 3, 7)])
def test_lists_of_pairs(K, rows, top, experts):
    rng = np.random.default_rng(rows + experts)
    chosen = np.stack([rng.permutation(experts)[:top] for _ in range(rows)]).astype(np.int32)
    lists = torch.full((experts, rows), -1, dtype=torch.int32, device="cuda:0")
    counts = torch.empty(experts, dtype=torch.int32, device="cuda:0")
    K.experts_group(dev(chosen), lists, counts)
    for e in range(experts):
        want = np.nonzero(chosen.reshape(-1) == e)[0]
        got = lists[e].cpu().numpy()
        assert int(counts[e]) == len(want) and np.array_equal(got[:len(want)], want) and (got[len(want):] == -1).all(), e
