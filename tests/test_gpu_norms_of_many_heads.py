"""Gated norms of a row's heads by pieces of 16 bytes, with each number of lanes a head may take, against float64."""

import pytest
import torch

from test_gpu_kernels import K      # noqa: F401  (the fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("after", [False, True])
@pytest.mark.parametrize("rows,groups,per,first", [(128, 17, 64, 0), (143, 16, 32, 8), (200, 33, 72, 16), (130, 16, 512, 8), (129, 5, 256, 8), (131, 15, 8, 0), (160, 4, 512, 8), (128, 2, 504, 8), (150, 3, 96, 4), (128, 6, 36, 2),
                                                  (130, 4, 128, 8), (128, 4, 136, 8), (129, 2, 256, 0), (128, 3, 264, 8), (130, 15, 64, 0), (131, 9, 72, 8), (128, 17, 128, 8), (129, 16, 136, 0),
                                                  (128, 16, 256, 8), (130, 16, 264, 0)])
def test_norms_of_many_heads(K, dtype, after, rows, groups, per, first):      # noqa: F811
    """Each number of lanes a group may take, with lanes and groups left over, in rows and in blocks; two that are not in pieces of 16 bytes; and
    both sides of the sizes up to which few groups have a wave each, and many 16 lanes."""
    g = torch.Generator().manual_seed(rows * per)
    width = groups * per
    y, z, w = torch.randn(rows, width, generator=g) * 3, torch.randn(rows, first + width + 8, generator=g).to(dtype), torch.rand(width, generator=g) + 0.5
    gate = torch.nn.functional.silu(z[:, first:first + width].double())
    values = y.double() if after else y.double() * gate
    grouped = values.view(rows, groups, per)
    want = (grouped / (grouped.square().mean(-1, keepdim=True) + 1e-5).sqrt()).view(rows, width) * w.double() * (gate if after else 1)
    outs = [torch.empty(rows, width, dtype=dtype, device="cuda:0")]
    if dtype == torch.bfloat16 and width % 32 == 0:
        outs.append(K.new_rows(rows, width, dtype, width, False))
    for out in outs:
        K.gated_group_rmsnorm(y.cuda(), z.cuda(), first, w.cuda(), 1e-5, out, groups, gate_after=after)
        got = out if isinstance(out, torch.Tensor) else K.from_blocked(out)
        assert float((got.double().cpu() - want).abs().max() / want.abs().max()) < (2 ** -8 if dtype == torch.bfloat16 else 2e-6)
