"""Norm, rotation and cache write of steps of many rows against float64: heads of one, two and four a thread, heads that leave lanes without one,
stretches of heads, and steps whose rows do not come out even with the workgroups of an XCD."""

import numpy as np
import pytest
import torch

from test_gpu_pudorax import dev, rounded

pytestmark = pytest.mark.gpu

PAGE, EPS = 64, 1e-5


@pytest.fixture(scope="module")
def K():
    from beholdd.kernels import HipKernels
    return HipKernels("cuda:0")


def turn(x, positions, freq, neighbours):
    """x [n, heads, dim] with its first 2 len(freq) dimensions turned, in pairs of neighbours or of halves; the angle is the float32 product."""
    half = len(freq)
    if not half:
        return x
    angle = (positions.astype(np.float32)[:, None] * freq.astype(np.float32)).astype(np.float64)[:, None, :]
    c, s, out = np.cos(angle), np.sin(angle), x.copy()
    one, two = (slice(0, 2 * half, 2), slice(1, 2 * half, 2)) if neighbours else (slice(0, half), slice(half, 2 * half))
    a, b = x[..., one], x[..., two]
    out[..., one], out[..., two] = a * c - b * s, b * c + a * s
    return out


def padded(x, pad):
    return np.concatenate([x, np.zeros((*x.shape[:2], pad - x.shape[2]))], axis=2)


def check(K, dtype, rows, heads, kv_heads, pad, q, k, v, run):
    """`run(positions, row_seq, q_out, pages, table)` for two sequences, and what it writes against q, k and v [rows, heads, size]."""
    lengths = [rows - rows // 3, rows // 3]
    counts = [-(-length // PAGE) for length in lengths]
    order = np.random.default_rng(rows).permutation(sum(counts)).astype(np.int32)
    table = np.zeros((2, max(counts)), np.int32)
    table[0, :counts[0]], table[1, :counts[1]] = order[:counts[0]], order[counts[0]:]
    row_seq = np.repeat(np.arange(2, dtype=np.int32), lengths)
    q_out = torch.full((rows, heads * pad), float("nan"), dtype=dtype, device="cuda:0")
    pages = [torch.full(shape, float("nan"), dtype=dtype, device="cuda:0") for shape in ((sum(counts), kv_heads, PAGE, pad), (sum(counts), kv_heads, pad, PAGE))]
    positions = np.concatenate([np.arange(length, dtype=np.int32) for length in lengths])
    run(dev(positions), dev(row_seq), q_out, pages, dev(table))
    # half a unit of bfloat16's 8 bits, or 24-bit roundings of a norm's factor, two products and a sum of two; sines of angles of up to 1,100
    # radians from float32's functions: 4 units in the last place of 1
    near = (2.0 ** -8 if dtype == torch.bfloat16 else 0.0) + 1e-5
    got = [q_out.view(rows, heads, pad).double().cpu().numpy()]
    if K.kv_order(dtype, pad) == 0:
        page, token = table[row_seq, positions // PAGE], positions % PAGE
        got += [pages[0].double().cpu().numpy()[page, :, token], pages[1].double().cpu().numpy()[page, :, :, token]]
    for one, want in zip(got, (q, k, v)):
        want = padded(want, pad)
        assert np.abs(one - want).max() <= near * np.abs(want).max()
        assert (one[want == 0] == 0).all()
    return positions


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
# few rows a head a thread (two stretches of it), many rows one, two and four; half a wave of lanes; heads beyond a thread's four, in stretches
@pytest.mark.parametrize("rows,heads,kv_heads,dim,vdim,pad,turned,neighbours", [
    (300, 32, 8, 128, 128, 128, 64, False), (257, 3, 1, 256, 256, 256, 256, False), (1100, 8, 4, 128, 128, 128, 128, False), (1100, 16, 4, 128, 120, 128, 32, True),
    (1030, 32, 8, 128, 128, 128, 128, False), (1100, 40, 20, 252, 256, 256, 8, False), (1025, 2, 1, 32, 32, 32, 32, False), (300, 4, 2, 64, 60, 64, 0, False),
    (300, 2, 1, 32, 32, 32, 32, False), (100, 8, 2, 64, 64, 64, 64, False)])      # (the last two go an element at a time)
def test_heads_normed_one_by_one(K, dtype, rows, heads, kv_heads, dim, vdim, pad, turned, neighbours):
    rng = np.random.default_rng(rows + heads)
    proj, x = rounded(rng.standard_normal((rows, (heads + kv_heads) * dim + kv_heads * vdim)), dtype)
    wq, wk = ((1 + 0.3 * rng.standard_normal(dim)).astype(np.float32) for _ in range(2))
    freq = np.array([1e4 ** (-2.0 * i / turned) for i in range(turned // 2)], np.float32)
    positions = np.concatenate([np.arange(n) for n in (rows - rows // 3, rows // 3)])
    split = (heads + kv_heads) * dim
    qk, v = x[:, :split].reshape(rows, heads + kv_heads, dim).astype(np.float64), x[:, split:].reshape(rows, kv_heads, vdim).astype(np.float64)
    qk = qk / np.sqrt((qk ** 2).mean(-1, keepdims=True) + EPS)
    q, k = (turn(part * w, positions, freq, neighbours) for part, w in ((qk[:, :heads], wq), (qk[:, heads:], wk)))

    def run(positions, row_seq, q_out, pages, table):
        K.head_norm_rope_write(dev(proj), 0, None, dev(wq), dev(wk), EPS, dev(freq) if turned else None, turned, positions, row_seq, q_out, *pages, table, heads, kv_heads,
                               dim, vdim, pad, True, neighbours=neighbours)

    check(K, dtype, rows, heads, kv_heads, pad, q, k, v, run)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
# one, two, four and eight pieces a thread, fewer pieces than a wave has lanes, rows of few (an element at a time)
@pytest.mark.parametrize("rows,heads,kv_heads,dim,vdim,pad,turned", [(300, 8, 2, 64, 64, 64, 64), (257, 12, 4, 128, 128, 128, 64), (520, 16, 4, 128, 124, 128, 128),
                                                                     (300, 40, 8, 128, 128, 128, 32), (1030, 2, 1, 28, 32, 32, 8), (100, 8, 2, 64, 64, 64, 64)])
def test_whole_projections_normed(K, dtype, rows, heads, kv_heads, dim, vdim, pad, turned):
    rng = np.random.default_rng(rows + heads)
    qkv = rng.standard_normal((rows, (heads + kv_heads) * dim + kv_heads * vdim)).astype(np.float32)
    wq, wk = ((1 + 0.3 * rng.standard_normal(n * dim)).astype(np.float32) for n in (heads, kv_heads))
    freq = np.array([1e4 ** (-2.0 * i / turned) for i in range(turned // 2)], np.float32)
    positions = np.concatenate([np.arange(n) for n in (rows - rows // 3, rows // 3)])
    x = qkv.astype(np.float64)
    q, k, v = x[:, :heads * dim], x[:, heads * dim:(heads + kv_heads) * dim], x[:, (heads + kv_heads) * dim:].reshape(rows, kv_heads, vdim)
    q, k = (turn((part / np.sqrt((part ** 2).mean(-1, keepdims=True) + EPS) * w).reshape(rows, -1, dim), positions, freq, True) for part, w in ((q, wq), (k, wk)))

    def run(positions, row_seq, q_out, pages, table):
        K.whole_norm_rope_write(dev(qkv), dev(wq), dev(wk), EPS, dev(freq), turned, positions, row_seq, q_out, *pages, table, heads, kv_heads, dim, vdim, pad, True)

    check(K, dtype, rows, heads, kv_heads, pad, q, k, v, run)
