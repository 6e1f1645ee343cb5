"""Attention of short prompts on both sides of the rule that sends a step to the kernel whose four waves share a page, against float64."""

import math

import pytest
import torch

from test_gpu_kernels import PAGE, K, Layout, attention_reference_rows, dev, make_cache, rel, stored      # noqa: F401  (K: the fixture)

pytestmark = pytest.mark.gpu


# heads, kv heads, head size, rows and pasts of the sequences, which kernel: eight and nine rows; fewer than 16 columns; four and five
# pages of few tiles; seven pages at 255 and 256 tiles, eight pages (whose keys may be split)
@pytest.mark.parametrize("n_heads,kv_heads,head_dim,news,pasts,shared", [
    (8, 2, 128, [8, 3], [0, 60], 0), (8, 2, 128, [9, 3], [0, 60], 1), (2, 2, 64, [15, 2], [3, 0], 0), (2, 2, 64, [16, 2], [3, 0], 1),
    (32, 8, 128, [100, 80, 73], [0, 0, 0], 1), (5, 1, 96, [40, 9], [216, 1], 1), (5, 1, 96, [40, 9], [217, 1], 0),
    (4, 4, 32, [1008], [0], 0), (15, 15, 32, [272, 1], [176, 0], 1), (15, 15, 32, [16, 16], [401, 0], 0), (16, 16, 64, [100, 64, 33], [348, 0, 5], 1),
    (16, 1, 256, [12, 130], [0, 100], 1), (4, 2, 160, [33, 1, 64], [7, 190, 64], 1)])
def test_attention_of_short_prompts(K, n_heads, kv_heads, head_dim, news, pasts, shared):
    dtype, scale = torch.bfloat16, 1 / math.sqrt(head_dim)
    lengths = [p + n for p, n in zip(pasts, news)]
    assert int(K.lib.bh_attention_bf16_writes_blocked(len(news), max(news), n_heads, kv_heads, max(lengths) - 1)) == shared
    kp, vp, table, keys, values = make_cache(len(lengths), lengths, kv_heads, head_dim, dtype, seed=head_dim + n_heads)
    for s, n in enumerate(lengths):      # nothing behind a sequence's last key may reach a sum
        if n % PAGE:
            kp[int(table[s, (n - 1) // PAGE]), :, n % PAGE:, :] = float("nan")
            vp[int(table[s, (n - 1) // PAGE]), :, :, n % PAGE:] = float("nan")
    kp, vp = stored(K, kp, vp)
    n_rows = sum(news)
    q = torch.randn(n_rows, n_heads * head_dim, generator=torch.Generator().manual_seed(n_rows)).to(dtype)
    positions = torch.tensor([p + t for p, n in zip(pasts, news) for t in range(n)], dtype=torch.int32)
    row_seq = torch.tensor([s for s, n in enumerate(news) for _ in range(n)], dtype=torch.int32)
    starts = [sum(news[:s]) for s in range(len(news) + 1)]
    layout = Layout(False, dev(torch.tensor(starts, dtype=torch.int32)), len(news), max(news), max(lengths) - 1)
    for window in (0, 50):
        out = torch.full((n_rows, n_heads * head_dim), float("nan"), dtype=dtype, device="cuda:0")
        blocks = K.to_blocked(out, block_rows=8 if n_rows <= 8 else 16) if (n_heads * head_dim) % 32 == 0 else None
        for to in (out, blocks):
            if to is not None:
                K.attention(dev(q), to, kp, vp, dev(table), dev(row_seq), dev(positions), n_heads, kv_heads, head_dim, scale, window, layout=layout)
        assert blocks is None or torch.equal(K.from_blocked(blocks), out)
        for s in range(len(news)):
            rows = slice(starts[s], starts[s + 1])
            want = attention_reference_rows(q[rows], keys[s], values[s], positions[rows], n_heads, kv_heads, head_dim, scale, window)
            assert rel(out[rows], want) < 8e-3, (s, window)      # probabilities and results of 8 bits


@pytest.mark.parametrize("cap,sloped,coef,every", [(0.0, False, 0.3, 7), (0.0, False, -0.6, 5), (0.0, True, 0.0, 0), (1.5, False, 0.0, 0), (1.5, True, 0.3, 7)])
@pytest.mark.parametrize("n_heads,kv_heads,head_dim,new", [(4, 2, 128, 200), (8, 1, 64, 5), (2, 2, 32, 700)])
def test_forms_of_scores(K, n_heads, kv_heads, head_dim, new, cap, sloped, coef, every):
    """A query's factor stays out of the scores where it cannot be negative, and is in them where it is for late positions; slopes; a cap."""
    dtype, scale, past = torch.bfloat16, 1 / math.sqrt(head_dim), 30
    kp, vp, table, keys, values = make_cache(1, [past + new], kv_heads, head_dim, dtype, seed=new)
    q = torch.randn(new, n_heads * head_dim, generator=torch.Generator().manual_seed(new)).to(dtype)
    positions = torch.arange(past, past + new, dtype=torch.int32)
    layout = Layout(False, dev(torch.tensor([0, new], dtype=torch.int32)), 1, new, past + new - 1)
    out = torch.full((new, n_heads * head_dim), float("nan"), dtype=dtype, device="cuda:0")
    kp, vp = stored(K, kp, vp)
    slopes = torch.linspace(0.0, 0.25, n_heads) if sloped else None
    K.attention(dev(q), out, kp, vp, dev(table), dev(torch.zeros(new, dtype=torch.int32)), dev(positions), n_heads, kv_heads, head_dim, scale, 0,
                layout=layout, softcap=cap, slopes=None if slopes is None else dev(slopes), q_temp=(coef, every) if every else None)
    factor = 1 + coef * torch.log(((positions + 1) // every).double() + 1) if every else torch.ones(new).double()
    scores = torch.einsum("nhd,khd->nhk", q.double().view(new, n_heads, head_dim) * factor[:, None, None],
                          keys[0].double().repeat_interleave(n_heads // kv_heads, 1)) * scale
    if cap:
        scores = cap * torch.tanh(scores / cap)
    gap = positions[:, None] - torch.arange(past + new)
    if sloped:
        scores = scores - slopes.double()[:, None] * gap[:, None, :]
    p = scores.masked_fill((gap < 0)[:, None, :], float("-inf")).softmax(-1)
    want = torch.einsum("nhk,khd->nhd", p, values[0].double().repeat_interleave(n_heads // kv_heads, 1)).reshape(new, -1)
    assert rel(out, want) < 8e-3                             # probabilities and results of 8 bits


@pytest.mark.parametrize("scale,coef,every", [(0.0, 0.3, 7), (0.0, 0.0, 0), (-0.2, 0.3, 7), (-0.2, 0.0, 0)])
@pytest.mark.parametrize("n_heads,kv_heads,head_dim,new,past", [(4, 2, 128, 200, 30), (8, 1, 64, 5, 30), (2, 2, 192, 1, 700)])
def test_scores_whose_factor_is_not_positive(K, n_heads, kv_heads, head_dim, new, past, scale, coef, every):
    """Nothing: the average of what is seen.  Negative: the smallest product has the largest score.  On the kernel of prompts, on the one of
    few rows, and with keys in splits; then the last row once more as a decode step from the projection rows."""
    dtype, length = torch.bfloat16, past + new
    kp, vp, table, keys, values = make_cache(1, [length], kv_heads, head_dim, dtype, seed=new)
    g = torch.Generator().manual_seed(new)
    q = torch.randn(new, n_heads * head_dim, generator=g).to(dtype)
    positions = torch.arange(past, length, dtype=torch.int32)
    kp, vp = stored(K, kp, vp)
    q_temp = (coef, every) if every else None
    factor = 1 + coef * torch.log(((positions + 1) // every).double() + 1) if every else torch.ones(new).double()
    scores = torch.einsum("nhd,khd->nhk", q.double().view(new, n_heads, head_dim) * factor[:, None, None],
                          keys[0].double().repeat_interleave(n_heads // kv_heads, 1)) * scale
    seen = positions[:, None] >= torch.arange(length)
    want = torch.einsum("nhk,khd->nhd", scores.masked_fill(~seen[:, None, :], float("-inf")).softmax(-1),
                        values[0].double().repeat_interleave(n_heads // kv_heads, 1)).reshape(new, -1)
    out = torch.full((new, n_heads * head_dim), float("nan"), dtype=dtype, device="cuda:0")
    layout = Layout(new == 1, dev(torch.tensor([0, new], dtype=torch.int32)), 1, new, length - 1)
    K.attention(dev(q), out, kp, vp, dev(table), dev(torch.zeros(new, dtype=torch.int32)), dev(positions), n_heads, kv_heads, head_dim, scale, 0,
                layout=layout, q_temp=q_temp)
    assert rel(out, want) < 8e-3                             # probabilities and results of 8 bits
    row = torch.cat([q[-1:], keys[0][-1:].reshape(1, -1), values[0][-1:].reshape(1, -1)], 1)
    one = torch.full((1, n_heads * head_dim), float("nan"), dtype=dtype, device="cuda:0")
    layout = Layout(True, dev(torch.tensor([0, 1], dtype=torch.int32)), 1, 1, length - 1)
    assert K.attention_decode_pairs(dev(row), 0, one, None, None, 0.0, None, None, dev(positions[-1:]), kp, vp, dev(table), n_heads, kv_heads, head_dim,
                                    scale, True, layout, q_temp=q_temp)
    assert rel(one, want[-1:]) < 8e-3
    if not every:      # the launch from whole fused rows has scaled products only, and leaves such steps to the two
        assert not K.attention_decode_fused(dev(row), one, None, None, 0.0, None, None, dev(positions[-1:]), kp, vp, dev(table), n_heads, kv_heads,
                                            head_dim, scale, 0, True, layout)


@pytest.mark.parametrize("n_heads,kv_heads,head_dim,new", [(16, 8, 128, 448), (8, 2, 128, 256), (8, 4, 64, 256)])
def test_error_is_that_of_pages_by_their_own_maximum(K, n_heads, kv_heads, head_dim, new):
    """Scores spread by two, whose maximum grows by a little from page to page.  What else runs at these sizes rounds a page's probabilities
    against the page's own maximum, so that the largest is a one, and sums them unrounded: the error against float64 is held to that
    one's and 2.5 % (three seeds; measured 0.99 to 1.01 of it, and 1.04 to 1.07 with probabilities of more than one)."""
    dtype, scale, error, bound = torch.bfloat16, head_dim ** -0.5, 0.0, 0.0
    positions = torch.arange(new, dtype=torch.int32)
    for seed in range(3):
        kp, vp, table, keys, values = make_cache(1, [new], kv_heads, head_dim, dtype, seed=seed)
        q = (2 * torch.randn(new, n_heads * head_dim, generator=torch.Generator().manual_seed(seed))).to(dtype)
        kp, vp = stored(K, kp, vp)
        out = torch.full((new, n_heads * head_dim), float("nan"), dtype=dtype, device="cuda:0")
        K.attention(dev(q), out, kp, vp, dev(table), dev(torch.zeros(new, dtype=torch.int32)), dev(positions), n_heads, kv_heads, head_dim, scale, 0,
                    layout=Layout(False, dev(torch.tensor([0, new], dtype=torch.int32)), 1, new, new - 1))
        spread = lambda x: x.double().repeat_interleave(n_heads // kv_heads, 1).transpose(0, 1)
        scores = q.double().view(new, n_heads, head_dim).transpose(0, 1) @ spread(keys[0]).transpose(1, 2) * scale
        scores = scores.masked_fill(positions[:, None] < positions, float("-inf"))
        value, total, top, sums = 0.0, 0.0, scores.amax(-1, keepdim=True), spread(values[0])
        for first in range(0, new, 64):
            page = scores[:, :, first:first + 64]
            own = page.amax(-1, keepdim=True).clamp_min(-1e30)
            p, factor = (page - own).exp(), (own - top).exp()
            value, total = value + p.to(dtype).double() @ sums[:, first:first + 64] * factor, total + p.sum(-1, keepdim=True) * factor
        rows = lambda x: x.transpose(0, 1).reshape(new, -1)
        want, other = rows(scores.softmax(-1) @ sums), rows(value / total).to(dtype).double()
        error, bound = error + float((out.double().cpu() - want).norm() / want.norm()), bound + float((other - want).norm() / want.norm())
    assert error < 1.025 * bound, error / bound
