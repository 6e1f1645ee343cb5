"""Norm, rotation and cache write of steps of many rows, whose kernels take four dimensions a thread, against the same rows in steps of few,
which go an element at a time: the same queries and pages, but for the order of a norm's sum of squares (32 bits, up to 4,096 terms: 1e-6;
one step of bfloat16 where that turns a rounding, 2^-8 of a value at most)."""

import numpy as np
import pytest
import torch

from test_gpu_pudorax import dev, rounded

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16]
PAGE, ROWS, FEW = 64, 300, 100      # rows for every compute unit and more; parts of them that are not


@pytest.fixture(scope="module")
def K():
    from beholdd.kernels import HipKernels
    return HipKernels("cuda:0")


def pages_of(dtype, kv_heads, pad):
    return [torch.full(shape, 7.0, dtype=dtype, device="cuda:0") for shape in ((6, kv_heads, PAGE, pad), (6, kv_heads, pad, PAGE))]


def same(got, want, dtype):
    for a, b in zip(got, want):
        a, b = a.float(), b.float()
        near = 4e-6 if dtype == torch.float32 else 2.0 ** -7
        assert bool(((a - b).abs() <= near * b.abs() + 1e-6).all())
        assert float((a - b).norm()) <= (1e-6 if dtype == torch.float32 else 2e-3) * float(b.norm())


def many_and_few(K, dtype, heads, kv_heads, pad, write):
    """`write(rows, positions, row_seq, q_out, pages, table)` on all rows at once and in parts."""
    table = dev(np.array([[4, 0, 5, 2, 1]], np.int32))
    out = []
    for size in (ROWS, FEW):
        q_out, pages = torch.empty(ROWS, heads * pad, dtype=dtype, device="cuda:0"), pages_of(dtype, kv_heads, pad)
        for lo in range(0, ROWS, size):
            rows = slice(lo, lo + size)
            write(rows, dev(np.arange(lo, lo + size, dtype=np.int32)), dev(np.zeros(size, np.int32)), q_out[rows], pages, table)
        out.append([q_out, *pages])
    same(*out, dtype)


# heads that fill their lanes and that do not, one and several stretches of them, turns of both forms over all and some dimensions, no turn, no
# norm, a norm without weights, values that are keys, a cache that is another layer's; sizes that are no whole pieces stay with the other kernel
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("heads,kv_heads,dim,vdim,pad,turned,form", [
    (32, 8, 128, 128, 128, 64, {}), (8, 2, 64, 64, 64, 64, dict(neighbours=True, magnitude=1.3)), (5, 1, 24, 32, 32, 8, {}), (36, 4, 100, 44, 128, 12, dict(neighbours=True)),
    (3, 3, 256, 200, 256, 256, {}), (6, 2, 64, 64, 64, 16, dict(unit_norm=True)), (6, 2, 96, 96, 128, 32, dict(unit_norm=True, values_are_keys=True)),
    (4, 4, 32, 32, 32, 0, dict(bare=True)), (7, 1, 128, 128, 128, 128, dict(write=False)), (4, 2, 60, 60, 64, 20, {}), (4, 2, 30, 30, 32, 8, {})])
@pytest.mark.parametrize("first,more", [(0, 0), (4, 8), (3, 1)])
def test_heads_normed_one_by_one(K, dtype, heads, kv_heads, dim, vdim, pad, turned, form, first, more):
    form = dict(form)
    write_kv, bare = form.pop("write", True), form.pop("bare", False)
    rng = np.random.default_rng(heads * dim + vdim)
    channels = (heads + kv_heads) * dim + (0 if form.get("values_are_keys") else kv_heads * vdim)
    proj = dev(rounded(rng.standard_normal((ROWS, first + channels + more)), dtype)[0])
    bias = dev(rng.standard_normal(channels).astype(np.float32)) if first != 4 else None
    wq, wk = (None, None) if bare or form.get("unit_norm") else (dev((1 + 0.3 * rng.standard_normal(dim)).astype(np.float32)) for _ in range(2))
    freq = dev(np.array([1e4 ** (-2.0 * i / turned) for i in range(turned // 2)], np.float32)) if turned else None

    def write(rows, positions, row_seq, q_out, pages, table):
        K.head_norm_rope_write(proj[rows].contiguous(), first, bias, wq, wk, 1e-5, freq, turned, positions, row_seq, q_out, *pages, table, heads, kv_heads, dim, vdim,
                               pad, write_kv, **form)

    many_and_few(K, dtype, heads, kv_heads, pad, write)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("heads,kv_heads,dim,vdim,pad,turned,write_kv", [(16, 4, 128, 128, 128, 64, True), (32, 8, 128, 128, 128, 128, True), (4, 4, 60, 64, 64, 6, True),
                                                                       (3, 1, 24, 40, 64, 0, True), (8, 2, 64, 64, 64, 64, False), (48, 24, 128, 128, 128, 64, True),
                                                                       (4, 2, 30, 30, 32, 8, True)])
def test_whole_projections_normed(K, dtype, heads, kv_heads, dim, vdim, pad, turned, write_kv):
    rng = np.random.default_rng(heads * dim + vdim)
    qkv = dev(rng.standard_normal((ROWS, (heads + kv_heads) * dim + kv_heads * vdim)).astype(np.float32))
    wq, wk = (dev((1 + 0.3 * rng.standard_normal(n * dim)).astype(np.float32)) for n in (heads, kv_heads))
    freq = dev(np.array([1e4 ** (-2.0 * i / turned) for i in range(turned // 2)], np.float32)) if turned else None

    def write(rows, positions, row_seq, q_out, pages, table):
        K.whole_norm_rope_write(qkv[rows].contiguous(), wq, wk, 1e-5, freq, turned, positions, row_seq, q_out, *pages, table, heads, kv_heads, dim, vdim, pad, write_kv)

    many_and_few(K, dtype, heads, kv_heads, pad, write)
