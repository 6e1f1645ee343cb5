"""Products of more than 128 rows of packed weights on every tile they are compiled for, at the tiles' edges, against float64."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    from beholdd.kernels import HipKernels
    return HipKernels()


def rel(got, want):
    got = got.double().cpu() if got.dtype != torch.float64 else got.cpu()
    return float((got - want).abs().max() / want.abs().max())


# rows, weight rows and k one beyond and one short of whole tiles, of whole steps in the ring (64 k are two), of parts and halves of K
SIZES = [(129, 1024, 1024), (129, 1040, 1088), (256, 1024, 1152), (257, 128, 128), (257, 144, 192), (383, 1008, 320),      # few tiles
         (2049, 2064, 1088), (2049, 2032, 1152), (2048, 2048, 2048),                                                      # 128 x 128, whole K and in halves
         (2096, 3088, 512), (2047, 4096, 640), (1025, 4112, 256),                                                         # 256 x 128
         (2049, 6128, 256), (251, 5120, 2048), (140, 7168, 1280), (700, 6160, 2048), (8193, 4080, 128)]                   # 256 rows, and parts of K


@pytest.mark.parametrize("m,n,k", SIZES)
def test_products_of_many_rows(K, m, n, k):
    """float32 with and without accumulation, bfloat16 and gated, from activations whose buffer holds NaN behind the last row; the
    bounds are those of a sum of k float32 products and of one bfloat16 rounding."""
    from beholdd.kernels.library import BlockedRows
    g = torch.Generator(device="cuda:0").manual_seed(m + n + k)
    a = torch.randn(m, k, generator=g, device="cuda:0").to(torch.bfloat16)
    w = (torch.randn(2 * n, k, generator=g, device="cuda:0") * 0.05).to(torch.bfloat16)
    plain, both = K.pack_weight(w[:n].contiguous()), K.pack_weight(w)
    in_blocks = BlockedRows(torch.full((BlockedRows.padded_rows(m, 16) * k,), float("nan"), dtype=torch.bfloat16, device="cuda:0"), m, k)
    K.to_blocked(a, in_blocks)
    want, up = (a.double() @ w[:n].double().t()).cpu(), (a.double() @ w[n:].double().t()).cpu()
    bound = 4 * math.sqrt(k) * 2.0 ** -24
    for x in (in_blocks, a):
        out = torch.full((m, n), float("nan"), dtype=torch.float32, device="cuda:0")
        K.gemm(x, plain, out)
        assert rel(out, want) < bound
    base = torch.randn(m, n, generator=g, device="cuda:0")
    total = base.clone()
    K.gemm(in_blocks, plain, total, accumulate=True)
    assert rel(total, want + base.double().cpu()) < bound
    rounded = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda:0")
    K.gemm(in_blocks, plain, rounded)
    assert rel(rounded, want) < 4e-3
    gated = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda:0")
    K.gemm_swiglu(in_blocks, both, gated)
    assert rel(gated, want / (1 + torch.exp(-want)) * up) < 6e-3
    if n % 32 == 0:
        blocked = K.new_rows(m, n, torch.bfloat16, n, False)
        K.gemm_swiglu(in_blocks, both, blocked)
        assert torch.equal(K.from_blocked(blocked) if isinstance(blocked, BlockedRows) else blocked, gated)


@pytest.mark.parametrize("m,n,k", [(251, 5120, 2048), (129, 1024, 1024), (2048, 2048, 2048), (300, 4096, 1088)])
def test_products_of_many_rows_and_the_norm_behind_them(K, m, n, k):
    """`gemm(..., then_norm=)`: the residual as without the norm bit for bit, and its norm within a bfloat16 rounding."""
    from beholdd.kernels.library import BlockedRows
    from beholdd.parts.base import NormRequest, ProductReader
    g = torch.Generator(device="cuda:0").manual_seed(m + n)
    a = torch.randn(m, k, generator=g, device="cuda:0").to(torch.bfloat16)
    packed = K.pack_weight((torch.randn(n, k, generator=g, device="cuda:0") * 0.05).to(torch.bfloat16))
    base, weight = torch.randn(m, n, generator=g, device="cuda:0"), 1 + 0.3 * torch.randn(n, generator=g, device="cuda:0")
    plain, residual = base.clone(), base.clone()
    K.gemm(a, packed, plain, accumulate=True)
    normed = K.gemm(a, packed, residual, accumulate=True, then_norm=NormRequest(weight, 1e-5, ProductReader(n)))
    assert torch.equal(plain, residual)
    got = residual.double()
    want = got / torch.sqrt((got ** 2).mean(-1, keepdim=True) + 1e-5) * weight.double()
    assert rel(K.from_blocked(normed) if isinstance(normed, BlockedRows) else normed, want.cpu()) < 4e-3
