"""Decode attention from the projection rows with keys in one to 64 splits, whose partial results groups of eight are combined from, and
with last splits of no page, one page and four beside the new key, against float64."""

import math

import pytest
import torch

from test_gpu_kernels import K, Layout, as_rows, attention_reference_rows, dev, make_cache, rel, stored      # noqa: F401  (K: the fixture)

pytestmark = pytest.mark.gpu


# 24 and 25 pages a workgroup of one that has a compute unit for itself, and one column and five of them
@pytest.mark.parametrize("heads,kv_heads,head_dim", [(4, 4, 32), (20, 4, 64), (4, 4, 128)])
@pytest.mark.parametrize("context", [24 * 64, 24 * 64 + 1])
def test_long_runs_of_pages(K, heads, kv_heads, head_dim, context):
    dtype, scale, lengths = torch.bfloat16, 1 / math.sqrt(head_dim), [context] + [1, 70] * 31 + [context // 2]
    n = len(lengths)
    assert int(K.lib.bh_attention_bf16_splits(n, 1, heads, kv_heads, context - 1)) == 1
    kp, vp, table, keys, values = make_cache(n, lengths, kv_heads, head_dim, dtype, seed=context)
    qkv = torch.randn(n, (heads + 2 * kv_heads) * head_dim, generator=torch.Generator().manual_seed(context)).to(dtype)
    positions = torch.tensor([length - 1 for length in lengths], dtype=torch.int32)
    layout = Layout(True, dev(torch.arange(n + 1, dtype=torch.int32)), n, 1, context - 1)
    k_pages, v_pages = stored(K, kp, vp)
    out = torch.full((n, heads * head_dim), float("nan"), dtype=dtype, device="cuda:0")
    assert K.attention_decode_fused(dev(qkv), out, None, None, 0.0, None, None, dev(positions), k_pages, v_pages, dev(table), heads, kv_heads,
                                    head_dim, scale, 0, True, layout)
    for s, length in enumerate(lengths):
        row = qkv[s].reshape(heads + 2 * kv_heads, head_dim)
        key, value = keys[s].clone(), values[s].clone()
        key[-1], value[-1] = row[heads:heads + kv_heads], row[heads + kv_heads:]
        want = attention_reference_rows(row[:heads].reshape(1, -1), key, value, positions[s:s + 1], heads, kv_heads, head_dim, scale, 0)
        assert rel(out[s:s + 1], want) < 8e-3, (s, length)      # probabilities and results of 8 bits


@pytest.mark.parametrize("heads,kv_heads,head_dim", [(2, 1, 128), (5, 1, 64), (4, 2, 256), (3, 3, 96)])
@pytest.mark.parametrize("context,bucket", [(1, 1), (447, 7), (449, 8), (512, 16), (1100, 20), (1024, 32), (2049, 33), (4000, 72), (9000, 144), (17000, 272)])
def test_decode_attention_in_splits(K, heads, kv_heads, head_dim, context, bucket):
    dtype, scale = torch.bfloat16, 1 / math.sqrt(head_dim)
    lengths = [context, max(context // 3, 1), 1]      # the new token stands at length - 1
    n = len(lengths)
    kp, vp, table, keys, values = make_cache(n, lengths, kv_heads, head_dim, dtype, seed=context)
    wide = torch.zeros(n, bucket, dtype=torch.int32)
    wide[:, :table.shape[1]] = table
    g = torch.Generator().manual_seed(context)
    qkv = torch.randn(n, (heads + 2 * kv_heads) * head_dim, generator=g).to(dtype)
    positions = torch.tensor([length - 1 for length in lengths], dtype=torch.int32)
    layout = Layout(True, dev(torch.arange(n + 1, dtype=torch.int32)), n, 1, bucket * 64 - 1)
    k_pages, v_pages = stored(K, kp, vp)
    for block_rows in (0, 8):
        if block_rows and (heads * head_dim) % 32:
            continue
        out = torch.full((n, heads * head_dim), float("nan"), dtype=dtype, device="cuda:0")
        to = K.to_blocked(out, block_rows=8) if block_rows else out
        assert K.attention_decode_fused(dev(qkv), to, None, None, 0.0, None, None, dev(positions), k_pages, v_pages, dev(wide), heads, kv_heads,
                                        head_dim, scale, 0, True, layout)
        got = K.from_blocked(to) if block_rows else to
        for s, length in enumerate(lengths):
            row = qkv[s].reshape(heads + 2 * kv_heads, head_dim)
            key, value = keys[s].clone(), values[s].clone()
            key[-1], value[-1] = row[heads:heads + kv_heads], row[heads + kv_heads:]
            want = attention_reference_rows(row[:heads].reshape(1, -1), key, value, positions[s:s + 1], heads, kv_heads, head_dim, scale, 0)
            assert rel(got[s:s + 1], want) < 8e-3, (s, length)      # probabilities and results of 8 bits


@pytest.mark.parametrize("heads,kv_heads,head_dim", [(2, 1, 128), (5, 1, 64), (4, 2, 192)])
@pytest.mark.parametrize("context,bucket", [(1, 1), (449, 8), (2049, 33), (17000, 272)])
def test_decode_attention_in_splits_norms_and_turns(K, heads, kv_heads, head_dim, context, bucket):
    """The same with heads that are normed and rotated on the way (by the fifth wave, or, of more than 128, by all four), the key that
    the cache gets among them."""
    dtype, scale, eps = torch.bfloat16, 1 / math.sqrt(head_dim), 1e-5
    lengths = [context, max(context // 3, 1), 1]
    n = len(lengths)
    kp, vp, table, keys, values = make_cache(n, lengths, kv_heads, head_dim, dtype, seed=context)
    wide = torch.zeros(n, bucket, dtype=torch.int32)
    wide[:, :table.shape[1]] = table
    g = torch.Generator().manual_seed(context)
    qkv = (3 * torch.randn(n, (heads + 2 * kv_heads) * head_dim, generator=g)).to(dtype)
    weights = [(1 + 0.2 * torch.randn(head_dim, generator=g)).to(dtype) for _ in range(2)]
    angles = torch.arange(bucket * 64, dtype=torch.float64)[:, None] / 1e4 ** (torch.arange(0, head_dim, 2, dtype=torch.float64) / head_dim)
    positions = torch.tensor([length - 1 for length in lengths], dtype=torch.int32)
    layout = Layout(True, dev(torch.arange(n + 1, dtype=torch.int32)), n, 1, bucket * 64 - 1)
    k_pages, v_pages = stored(K, kp, vp)
    out = torch.full((n, heads * head_dim), float("nan"), dtype=dtype, device="cuda:0")
    assert K.attention_decode_fused(dev(qkv), out, dev(weights[0]), dev(weights[1]), eps, dev(angles.cos().float()), dev(angles.sin().float()),
                                    dev(positions), k_pages, v_pages, dev(wide), heads, kv_heads, head_dim, scale, 0, True, layout)
    k_rows, v_rows = as_rows(K, k_pages, v_pages)
    for s, length in enumerate(lengths):
        row = qkv[s].double().reshape(heads + 2 * kv_heads, head_dim)
        made = []
        for x, weight in ((row[:heads], weights[0]), (row[heads:heads + kv_heads], weights[1])):
            x = x / (x.square().mean(-1, keepdim=True) + eps).sqrt() * weight.double()
            low, high, cos, sin = x[:, :head_dim // 2], x[:, head_dim // 2:], angles[length - 1].cos(), angles[length - 1].sin()
            made.append(torch.cat([low * cos - high * sin, high * cos + low * sin], 1).to(dtype))
        key, value = keys[s].clone(), values[s].clone()
        key[-1], value[-1] = made[1], qkv[s].reshape(-1, head_dim)[heads + kv_heads:]
        page, token = int(wide[s, (length - 1) // 64]), (length - 1) % 64
        assert rel(k_rows[page, :, token], made[1]) < 8e-3 and torch.equal(v_rows[page, :, :, token].to(dtype), value[-1])
        want = attention_reference_rows(made[0].reshape(1, -1), key, value, positions[s:s + 1], heads, kv_heads, head_dim, scale, 0)
        assert rel(out[s:s + 1], want) < 8e-3, (s, length)      # probabilities and results of 8 bits


# keys in splits; more workgroups than compute units; heads of more than 128.  The last factor is negative from position 189 on.
@pytest.mark.parametrize("heads,kv_heads,head_dim,n,context", [(4, 2, 128, 2, 3000), (32, 8, 128, 40, 150), (4, 2, 192, 2, 900), (4, 2, 64, 1, 40)])
@pytest.mark.parametrize("coef,every", [(0.4, 16), (-0.3, 7)])
def test_a_factor_of_the_query_alone_in_one_launch(K, heads, kv_heads, head_dim, n, context, coef, every):
    dtype, scale = torch.bfloat16, 1 / math.sqrt(head_dim)
    lengths = [context - 3 * s for s in range(n)]
    kp, vp, table, keys, values = make_cache(n, lengths, kv_heads, head_dim, dtype, seed=context)
    qkv = torch.randn(n, (heads + 2 * kv_heads) * head_dim, generator=torch.Generator().manual_seed(context)).to(dtype)
    positions = torch.tensor([length - 1 for length in lengths], dtype=torch.int32)
    layout = Layout(True, dev(torch.arange(n + 1, dtype=torch.int32)), n, 1, context - 1)
    k_pages, v_pages = stored(K, kp, vp)
    out = torch.full((n, heads * head_dim), float("nan"), dtype=dtype, device="cuda:0")
    assert K.attention_decode_pairs(dev(qkv), 0, out, None, None, 0.0, None, None, dev(positions), k_pages, v_pages, dev(table), heads, kv_heads,
                                    head_dim, scale, True, layout, q_temp=(coef, every))
    for s, length in enumerate(lengths):
        row = qkv[s].reshape(heads + 2 * kv_heads, head_dim)
        key, value = keys[s].clone(), values[s].clone()
        key[-1], value[-1] = row[heads:heads + kv_heads], row[heads + kv_heads:]
        factor = 1 + coef * math.log(length // every + 1)
        want = attention_reference_rows(row[:heads].double().reshape(1, -1) * factor, key, value, positions[s:s + 1], heads, kv_heads, head_dim, scale, 0)
        assert rel(out[s:s + 1], want) < 8e-3, (s, length)


def test_splits_that_are_not_combined_are_refused_before_anything_runs(K):
    """65 splits of a decode step that writes its new key: an error, and cache and output as they were."""
    from beholdd.kernels import KernelError
    heads, kv_heads, head_dim, n_splits, length = 2, 1, 64, 65, 65 * 64
    kp, vp, table, _, _ = make_cache(1, [length], kv_heads, head_dim, torch.bfloat16, seed=1)
    k_pages, v_pages = stored(K, kp, vp)
    before = k_pages.clone(), v_pages.clone()
    rows = torch.ones(1, (heads + 2 * kv_heads) * head_dim, dtype=torch.bfloat16, device="cuda:0")
    out = torch.full((1, heads * head_dim), 7.0, dtype=torch.bfloat16, device="cuda:0")
    part_o, part_ml = torch.zeros(heads * n_splits * head_dim, device="cuda:0"), torch.zeros(heads * n_splits * 2, device="cuda:0")
    table, positions = dev(table), torch.tensor([length - 1], dtype=torch.int32, device="cuda:0")
    starts = torch.tensor([0, 1], dtype=torch.int32, device="cuda:0")
    with pytest.raises(KernelError, match="65 splits"):
        K._check(K.lib.bh_attention_decode_fused(
            rows.data_ptr(), out.data_ptr(), part_o.data_ptr(), part_ml.data_ptr(), k_pages.data_ptr(), v_pages.data_ptr(), table.data_ptr(),
            table.shape[1], positions.data_ptr(), starts.data_ptr(), 1, heads, kv_heads, head_dim, 0.125, 0, length - 1, n_splits, None, None, 0,
            0.0, None, None, 0, 0, 1, 0, K._stream()))
    assert torch.equal(k_pages, before[0]) and torch.equal(v_pages, before[1]) and bool((out == 7.0).all())


@pytest.mark.parametrize("heads,kv_heads,head_dim,context,new", [(4, 2, 128, 300, 1), (3, 3, 96, 300, 1), (4, 2, 256, 40, 1), (4, 2, 128, 60, 5), (4, 2, 64, 90, 40),
                                                                 (4, 2, 128, 0, 300)])
def test_attention_into_rows_that_stand_on_two_bytes(K, heads, kv_heads, head_dim, context, new):
    """Decode steps, short steps and prompts that would else go to the kernel whose stores are 8 bytes: what lies around is as it was."""
    dtype, scale, length = torch.bfloat16, 1 / math.sqrt(head_dim), context + new
    kp, vp, table, keys, values = make_cache(1, [length], kv_heads, head_dim, dtype, seed=length)
    k_pages, v_pages = stored(K, kp, vp)
    q = torch.randn(new, heads * head_dim, generator=torch.Generator().manual_seed(length)).to(dtype)
    positions = torch.arange(context, length, dtype=torch.int32)
    want = attention_reference_rows(q, keys[0], values[0], positions, heads, kv_heads, head_dim, scale, 0)
    layout = Layout(new == 1, dev(torch.tensor([0, new], dtype=torch.int32)), 1, new, length - 1)
    for shift in (1, 2, 3):
        space = torch.full((q.numel() + 8,), 7.0, dtype=dtype, device="cuda:0")
        out = space[shift:shift + q.numel()].view(new, heads * head_dim)
        K.attention(dev(q), out, k_pages, v_pages, dev(table), dev(torch.zeros(new, dtype=torch.int32)), dev(positions), heads, kv_heads, head_dim,
                    scale, 0, layout=layout)
        assert rel(out, want) < 8e-3                             # probabilities and results of 8 bits
        assert bool((space[:shift] == 7.0).all()) and bool((space[shift + q.numel():] == 7.0).all())
    if new == 1:
        row = torch.cat([q, keys[0][-1:].reshape(1, -1), values[0][-1:].reshape(1, -1)], 1)
        assert K.attention_decode_fused(dev(row), out, None, None, 0.0, None, None, dev(positions), k_pages, v_pages, dev(table), heads, kv_heads,
                                        head_dim, scale, 0, True, layout)
        assert rel(out, want) < 8e-3
