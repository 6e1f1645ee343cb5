"""The gated norm in pieces of four columns against float64: one piece, rows that fill one to four pieces a thread, the widest row that is
held and one beyond it, and gates that do not lie on a piece."""

import pytest
import torch

from test_gpu_kernels import K, dev      # noqa: F401  (K: the fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,width,offset", [(1, 4, 4), (65, 1028, 0), (16, 4096, 8), (130, 8192, 0), (3, 16384, 4), (2, 16388, 0), (20, 256, 3)])
def test_gated_rmsnorm_in_pieces(K, dtype, rows, width, offset):
    g = torch.Generator().manual_seed(rows + width)
    o, proj, w = torch.randn(rows, width, generator=g) * 3, (torch.randn(rows, offset + width, generator=g) * 2).to(dtype), torch.randn(width, generator=g)
    out = torch.full((rows, width), float("nan"), dtype=dtype, device="cuda:0")
    K.gated_rmsnorm(dev(o), dev(proj), offset, dev(w), 1e-6, out)
    want = o.double() * torch.rsqrt(o.double().square().mean(1, keepdim=True) + 1e-6) * w.double() * torch.sigmoid(proj[:, offset:].double())
    # a sum of `width` squares, and a handful of roundings to 24 bits; the result's own rounding
    bound = ((width ** 0.5 + 8) * 2.0 ** -23 + (2.0 ** -8 if dtype == torch.bfloat16 else 0.0)) * want.abs() + 1e-30
    assert bool(((out.cpu().double() - want).abs() <= bound).all())
