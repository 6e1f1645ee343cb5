"""A small matrix per head on the matrix cores against float64: tiles of rows and of outputs that are not full, outputs in blocks, and
slices that do not lie on 16 bytes (which the kernel for every size takes)."""

import pytest
import torch

from test_gpu_kernels import K, dev      # noqa: F401  (K: the fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,heads,n_in,n_out,x_first,y_first", [
    (1, 3, 32, 16, 0, 0), (16, 2, 128, 192, 8, 0), (17, 4, 192, 128, 0, 4), (300, 2, 256, 272, 0, 0), (70, 1, 224, 48, 16, 8), (33, 5, 160, 80, 0, 0),
    (2050, 8, 128, 192, 0, 64), (40, 2, 64, 64, 3, 0), (40, 2, 64, 64, 0, 2)])
def test_heads_in_tiles(K, rows, heads, n_in, n_out, x_first, y_first):
    g = torch.Generator().manual_seed(rows + n_in)
    x_head, y_head = n_in + x_first + 8 - x_first % 8, n_out + y_first + (8 if y_first else 0)
    x = torch.randn(rows, heads * x_head, generator=g).bfloat16()
    w = (torch.randn(heads, n_in, n_out, generator=g) / n_in ** 0.5).bfloat16()
    y = torch.full((rows, heads * y_head), 9.0, dtype=torch.bfloat16, device="cuda:0")
    K.heads_linear(dev(x), x_head, x_first, dev(w), y, y_head, y_first, heads)
    got = y.cpu().double().view(rows, heads, y_head)
    inputs = x.double().view(rows, heads, x_head)[:, :, x_first:x_first + n_in]
    want = torch.einsum("rhi,hio->rho", inputs, w.double())
    # exact products, 32-bit sums, one rounding to 8 bits
    bound = 2.0 ** -8 * want.abs() + n_in * 2.0 ** -23 * torch.einsum("rhi,hio->rho", inputs.abs(), w.double().abs())
    assert bool(((got[:, :, y_first:y_first + n_out] - want).abs() <= bound).all())
    assert bool((got[:, :, :y_first] == 9.0).all()) and bool((got[:, :, y_first + n_out:] == 9.0).all())
    if (heads * y_head) % 32 == 0 and y_first == 0 and y_head == n_out:
        out = K.to_blocked(torch.full_like(y, float("nan")))
        K.heads_linear(dev(x), x_head, x_first, dev(w), out, y_head, 0, heads)
        assert torch.equal(K.from_blocked(out), y)
