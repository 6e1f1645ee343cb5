"""Residual streams and the squared ReLU in 16-byte pieces, against float64: one to four streams and more than that, widths around a
workgroup's threads, rows that do not lie on 16 bytes."""

import pytest
import torch

from test_gpu_kernels import K, dev      # noqa: F401  (K: the fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,streams,width,apart", [(1, 1, 4, 0), (3, 2, 4096, 0), (70, 2, 2048, 0), (64, 3, 1028, 0), (65, 4, 8192, 0), (2, 4, 8192, 0),
                                                      (64, 1, 8192, 0), (5, 2, 8196, 0), (3, 5, 64, 0), (66, 2, 1024, 1), (2, 2, 30, 0)])
def test_streams_update_and_norm(K, dtype, rows, streams, width, apart):
    g = torch.Generator().manual_seed(rows + streams + width)
    x, y = torch.randn(rows, streams, width, generator=g), torch.randn(rows, width, generator=g)
    mix, give, take = torch.randn(streams, streams, generator=g), torch.randn(streams, generator=g), torch.randn(streams, generator=g)
    scale, weight = torch.randn(width, generator=g), torch.randn(width, generator=g)
    new = torch.einsum("rsw,st->rtw", x.double(), mix.double()) + give.double()[:, None] * (scale.double() * y.double())[:, None]
    size = (x.double().abs().sum(1) * mix.double().abs().max() + (scale * y).double().abs() * give.double().abs().max()).max()
    for whole in (False, True):
        held = torch.empty(x.numel() + 4, device="cuda:0")[apart:apart + x.numel()].view(x.shape)      # apart: 4 bytes off
        held.copy_(x)
        out = torch.empty(rows, width, dtype=dtype, device="cuda:0")
        if whole:
            K.streams_update_rmsnorm(held, dev(y), dev(mix), dev(give), dev(scale), dev(take), dev(weight), 1e-6, out)
        else:
            K.streams_update(held, dev(y), dev(mix), dev(give), dev(scale))
        assert float((held.cpu().double() - new).abs().max()) <= (streams + 3) * 2.0 ** -24 * float(size)
    u = torch.einsum("rtw,t->rw", new, take.double())
    want = u / torch.sqrt((u * u).mean(-1, keepdim=True) + 1e-6) * weight.double()
    # the sum of the streams may cancel: its error is absolute, the rounding of the result relative
    slack = 64 * 2.0 ** -24 * float(size) * float(take.abs().sum()) / float(torch.sqrt((u * u).mean(-1)).min()) * float(weight.abs().max())
    assert float(((out.cpu().double() - want).abs() - (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -20) * want.abs()).max()) <= slack


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,width,blocked", [(1, 8, 0), (3, 4104, 0), (17, 2048, 16), (5, 96, 8), (2, 33, 0), (70, 64, 16)])
def test_squared_relu(K, dtype, rows, width, blocked):
    g = torch.Generator().manual_seed(width)
    x = (torch.randn(rows, width, generator=g) * 3).to(dtype)
    want = torch.relu(x.float()).square().to(dtype)
    assert torch.equal(_in_place(K, dev(x)), want)
    if blocked and dtype == torch.bfloat16:
        out = K.to_blocked(dev(x), block_rows=blocked)
        K.relu_squared(dev(x), out)
        assert torch.equal(K.from_blocked(out).cpu(), want)


def _in_place(K, x):
    K.relu_squared(x)
    return x.cpu()
