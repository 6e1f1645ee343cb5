"""Recurrences with a scalar decay as products, at the sizes where a workgroup's pieces and a wave's columns of a state change: the widest
keys, values of more than eight columns of tiles and of no power of two, heads that share keys in groups that fill no round of XCDs."""

import pytest
import torch

from test_gpu_decay_scan import test_lightning_scan_as_products as lightning, test_state_space_scan_as_products as state_space
from test_gpu_kernels import K      # noqa: F401  (the fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,dim,vdim,lengths", [(1, 288, 16, [700]), (16, 64, 256, [1500, 1, 70]), (3, 96, 144, [1100, 64, 65]),
                                                    (9, 160, 112, [300, 130]), (5, 128, 128, [63, 1, 1000])])
def test_lightning_sizes(K, heads, dim, vdim, lengths):
    lightning(K, torch.bfloat16, heads, dim, vdim, [0.5 + 0.5 * (i + 1) / (heads + 1) for i in range(heads)], lengths)


@pytest.mark.parametrize("heads,groups,vdim,n_state,lengths", [(12, 4, 80, 128, [900, 3]), (14, 2, 128, 64, [65, 500]), (64, 1, 64, 128, [1300, 700]),
                                                               (24, 8, 64, 160, [640, 64])])
def test_state_space_sizes(K, heads, groups, vdim, n_state, lengths):
    state_space(K, torch.bfloat16, heads, groups, vdim, n_state, (-1.0, 2.0), lengths)
