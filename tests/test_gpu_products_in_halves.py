"""Products of 33 to 128 rows whose workgroups cut their k in two: every number of row blocks, one part and several, a last part that is shorter,
weight rows that leave waves idle, and the sizes on both sides of the rule, against products in 64 bits of the same bfloat16 operands
(32-bit sums of up to 4,096 products: 1e-6 of the result and less)."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    from beholdd.kernels import HipKernels
    return HipKernels("cuda:0")


@pytest.mark.parametrize("rows", [33, 48, 49, 64, 96, 97, 128])
@pytest.mark.parametrize("outputs,k", [(128, 512), (144, 768), (1024, 1024), (1040, 2816), (2048, 2048), (4096, 512), (4112, 2048), (16400, 512)])
@pytest.mark.parametrize("accumulate", [False, True])
def test_products_cut_within_their_workgroups(K, rows, outputs, k, accumulate):
    generator = torch.Generator().manual_seed(rows * outputs + k)
    a = torch.randn(rows, k, generator=generator).bfloat16().to("cuda:0")
    w = (0.05 * torch.randn(outputs, k, generator=generator)).bfloat16().to("cuda:0")
    held = torch.randn(rows, outputs, generator=generator).to("cuda:0")
    out = held.clone()
    K.gemm(a, K.pack_weight(w), out, accumulate=accumulate)
    want = a.double() @ w.double().t() + (held.double() if accumulate else 0.0)
    assert float((out.double() - want).norm() / want.norm()) < 1e-6
    assert float((out.double() - want).abs().max() / want.abs().max()) < 1e-5
