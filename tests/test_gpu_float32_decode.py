"""Float32 decode attention from the projection rows (norm, rotation, cache write and attention in one launch) against float64 and against
the two launches it takes the place of."""

import math

import pytest
import torch

from test_gpu_kernels import K, Layout, attention_reference_rows, dev, make_cache      # noqa: F401  (K: the fixture)

pytestmark = pytest.mark.gpu


# lengths: position 0, a page's first and last slots, one page a wave and more; one wave a row (a page; few pages of many rows), four and eight
@pytest.mark.parametrize("lengths", [[1], [64, 1, 63], [65, 128, 129, 1, 64], [40 + i % 200 for i in range(300)], [700, 3, 1025, 257]])
@pytest.mark.parametrize("with_norm,with_rope,write_kv,window", [(True, True, True, 0), (False, False, True, 0), (True, False, True, 70), (False, True, True, 1),
                                                                 (True, True, False, 0), (True, True, False, 64)])
@pytest.mark.parametrize("heads,kv_heads,head_dim", [(8, 4, 128), (3, 3, 64), (6, 1, 256), (4, 2, 96), (2, 1, 32), (4, 1, 160)])
def test_float32_decode_attention_from_the_projection_rows(K, heads, kv_heads, head_dim, with_norm, with_rope, write_kv, window, lengths):
    if with_rope and head_dim % 64:
        with_rope = False
    n, eps, scale = len(lengths), 1e-5, 1 / math.sqrt(head_dim)
    kp, vp, table, keys, values = make_cache(n, lengths, kv_heads, head_dim, torch.float32, seed=head_dim + n)
    g = torch.Generator().manual_seed(head_dim + n)
    qkv = torch.randn(n, (heads + 2 * kv_heads) * head_dim, generator=g)
    qw, kw = (1 + 0.2 * torch.randn(head_dim, generator=g) for _ in range(2))
    freqs = 1.0 / 10000.0 ** (torch.arange(0, head_dim, 2, dtype=torch.float64) / head_dim)
    angles = torch.arange(1100, dtype=torch.float64)[:, None] * freqs
    cos, sin = angles.cos().float(), angles.sin().float()
    positions = torch.tensor([length - 1 for length in lengths], dtype=torch.int32)
    layout = Layout(True, dev(torch.arange(n + 1, dtype=torch.int32)), n, 1, max(lengths) - 1)
    weights = (dev(qw), dev(kw)) if with_norm else (None, None)
    tables = (dev(cos), dev(sin)) if with_rope else (None, None)
    one, two = (torch.full((n, heads * head_dim), float("nan"), device="cuda:0") for _ in range(2))
    k_one, v_one, k_two, v_two = dev(kp), dev(vp), dev(kp), dev(vp)
    if write_kv:      # where the new key and value go, nothing finite stands before
        for s, p in enumerate(positions.tolist()):
            for k_pages, v_pages in ((k_one, v_one), (k_two, v_two)):
                k_pages[int(table[s, p // 64]), :, p % 64] = float("nan")
                v_pages[int(table[s, p // 64]), :, :, p % 64] = float("inf")
    rows, row_seq = dev(qkv), dev(torch.arange(n, dtype=torch.int32))
    assert K.attention_decode_fused(rows, one, *weights, eps, *tables, dev(positions), k_one, v_one, dev(table), heads, kv_heads, head_dim,
                                    scale, window, write_kv, layout) is True
    q = torch.empty_like(two)
    K.qk_norm_rope_cache(rows, q, *weights, eps, *tables, dev(positions), row_seq, k_two, v_two, dev(table), heads, kv_heads, head_dim, write_kv, max(lengths) - 1)
    K.attention(q, two, k_two, v_two, dev(table), row_seq, dev(positions), heads, kv_heads, head_dim, scale, window, layout=layout)
    assert torch.equal(v_one, v_two)
    assert bool(((k_one - k_two).abs() <= 2.0 ** -20 * k_two.abs().max()).all())      # sums of squares in another order

    def made(x, w, pos):      # norm and rotation in 64 bits
        x = x.double()
        if with_norm:
            x = x / (x.square().mean(-1, keepdim=True) + eps).sqrt() * w.double()
        if with_rope:
            a, b, half = x[..., :head_dim // 2], x[..., head_dim // 2:], angles[pos]
            x = torch.cat((a * half.cos() - b * half.sin(), a * half.sin() + b * half.cos()), -1)
        return x

    for s in range(0, n, 1 if n < 10 else 37):
        pos, row = int(positions[s]), qkv[s].reshape(heads + 2 * kv_heads, head_dim)
        key, value = keys[s].double(), values[s].double()
        if write_kv:
            key[pos], value[pos] = made(row[heads:heads + kv_heads], kw, pos), row[heads + kv_heads:].double()
        want = attention_reference_rows(made(row[:heads], qw, pos).reshape(1, -1), key, value, positions[s:s + 1].long(), heads, kv_heads, head_dim, scale, window)
        for got in (one, two):
            # 64 roundings each of a score of a few units, of a probability and of a sum of at most ~1,000 values of at most ~5
            assert float((got[s].cpu().double() - want.reshape(-1)).abs().max()) < 64 * 2.0 ** -24 * 10, (s, pos)


def test_float32_decode_attention_says_when_it_cannot(K):
    kp, vp, table, _, _ = make_cache(2, [10, 70], 2, 64, torch.float32, seed=1)
    positions, layout = dev(torch.tensor([9, 69], dtype=torch.int32)), Layout(True, dev(torch.arange(3, dtype=torch.int32)), 2, 1, 69)
    store = torch.randn(2 * 8 * 64 + 1, device="cuda:0")
    out, cos = torch.empty(2, 256, device="cuda:0"), torch.randn(80, 16, device="cuda:0")
    weight = torch.ones(64, device="cuda:0", dtype=torch.bfloat16)

    def asked(rows, qw=None, tables=(None, None), step=layout):
        return K.attention_decode_fused(rows, out, qw, qw, 1e-5, *tables, positions, dev(kp), dev(vp), dev(table), 4, 2, 64, 0.1, 0, True, step)

    rows = store[:1024].view(2, 512)
    assert asked(rows) is True
    assert asked(store[1:].view(2, 512)) is False                    # rows that are not on 16 bytes
    assert asked(rows, qw=weight) is False                           # weights of another type
    assert asked(rows, tables=(cos, cos)) is False                   # a rotation of half of the head
    assert asked(rows, step=Layout(True, layout.seq_start, 1, 2, 69)) is False


@pytest.mark.parametrize("lengths,news", [([1, 64, 33], 1), ([2, 63], 2), ([64] * 3, 3)])
@pytest.mark.parametrize("heads,kv_heads,head_dim", [(8, 4, 128), (4, 2, 96), (4, 2, 64), (2, 1, 160)])
def test_float32_rows_of_one_page_whatever_the_step_may_see(K, heads, kv_heads, head_dim, lengths, news):
    """A captured step is launched for more pages than its rows hold: the results are, bit for bit, those of a launch that knows how few."""
    n, width = len(lengths), (heads + 2 * kv_heads) * head_dim
    kp, vp, table, _, _ = make_cache(n, lengths, kv_heads, head_dim, torch.float32, seed=head_dim + n)
    g = torch.Generator().manual_seed(head_dim)
    positions = torch.cat([torch.arange(max(length - news, 0), length) for length in lengths]).int()
    counts = [min(news, length) for length in lengths]
    rows = sum(counts)
    row_seq = torch.repeat_interleave(torch.arange(n), torch.tensor(counts)).int()
    start = torch.tensor([0] + counts).cumsum(0).int()
    q, qkv = torch.randn(rows, heads * head_dim, generator=g), torch.randn(rows, width, generator=g)
    results = []
    for furthest in (63, 1023):
        out = torch.full((rows, heads * head_dim), float("nan"), device="cuda:0")
        layout = Layout(news == 1, dev(start), n, news, furthest)
        K.attention(dev(q), out, dev(kp), dev(vp), dev(table), dev(row_seq), dev(positions), heads, kv_heads, head_dim, 0.1, 0, layout=layout)
        results.append([out])
        if news == 1:
            out, k_pages, v_pages = torch.full_like(out, float("nan")), dev(kp), dev(vp)
            assert K.attention_decode_fused(dev(qkv), out, None, None, 1e-5, None, None, dev(positions), k_pages, v_pages, dev(table), heads, kv_heads,
                                            head_dim, 0.1, 0, True, layout) is True
            results[-1] += [out, k_pages, v_pages]
    assert all(torch.equal(a, b) and not a.isnan().any() for a, b in zip(*results))
