"""Decode attention from the projection rows with keys in one to 64 splits, whose partial results groups of eight are combined from, and
with last splits of no page, one page and four beside the new key, against float64; and the embedding at widths of whole and cut pieces."""

import math

import pytest
import torch

from test_gpu_kernels import K, Layout, attention_reference_rows, dev, make_cache, rel, stored      # noqa: F401  (K: the fixture)

pytestmark = pytest.mark.gpu


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


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width", [4, 6, 1020, 1024, 1028, 4100, 5120])
def test_embedding_rows(K, dtype, width):
    table = torch.randn(50, width, generator=torch.Generator().manual_seed(width)).to(dtype).cuda()
    tokens = torch.tensor([3, 49, 0, -1, 50, 17, 17], dtype=torch.int32, device="cuda:0")      # ids outside the table read row 0
    source = torch.tensor([-1, -1, 1, -1, -1, 0, -1], dtype=torch.int32, device="cuda:0")
    fed = torch.tensor([8, 9], dtype=torch.int32, device="cuda:0")
    out = torch.full((7, width), float("nan"), device="cuda:0")
    K.embed(tokens, table, out)
    assert torch.equal(out, table.float()[[3, 49, 0, 0, 0, 17, 17]])
    K.embed(tokens, table, out, token_src=source, fed_tokens=fed)
    assert torch.equal(out, table.float()[[3, 49, 9, 0, 0, 8, 17]])
