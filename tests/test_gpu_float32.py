"""The float32 engine's own kernels (products and attention) against float64, where their tiles, slices and pages end."""

import math

import pytest
import torch

from test_gpu_kernels import K, Layout, attention_reference_rows, dev, make_cache    # noqa: F401  (K: the fixture)

pytestmark = pytest.mark.gpu


def product_bound(a, w, k):
    """Elementwise: a sum of k products in blocks.  A lane's chain is at most k / 16 products long (few rows), a slice's 32 and then
    k / 32 slices (many rows); 64 more roundings cover the additions over blocks, waves and into the result."""
    return (k / 16 + 64) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T)


# rows: around the groups of four, the last of the few, the tiles; outputs: one, tile remainders, both splits of a workgroup's
# rows; K: shorter than a load of the wave, remainders of a chunk of 64 and of a slice of 32, long enough for eight waves
@pytest.mark.parametrize("m,n,k", [(1, 1, 4), (1, 5, 60), (3, 64, 64), (4, 1030, 1024), (5, 7, 68), (8, 4099, 256), (9, 130, 516),
                                   (16, 8200, 132), (17, 33, 2052), (31, 516, 4096), (32, 16, 2048), (33, 65, 36), (64, 64, 32),
                                   (65, 300, 100), (130, 4, 1028), (257, 640, 260), (2050, 2100, 64), (2048, 2049, 132)])
def test_float32_products(K, m, n, k):
    g = torch.Generator().manual_seed(m + n + k)
    a, w, c = torch.randn(m, k, generator=g), torch.randn(n, k, generator=g), torch.randn(m, n, generator=g)
    want = a.double() @ w.double().T
    out = torch.full((m, n), float("nan"), device="cuda:0")
    K.gemm(dev(a), dev(w), out)
    assert bool(((out.cpu().double() - want).abs() <= product_bound(a, w, k)).all())
    summed = dev(c)
    K.gemm(dev(a), dev(w), summed, accumulate=True)
    assert bool(((summed.cpu().double() - want - c).abs() <= product_bound(a, w, k) + 2.0 ** -24 * (want.abs() + c.abs() + 1)).all())


# slices of 32 k: one to nine for waves that own 64 x 64 outputs, the same for two (K a multiple of 64) and four (of 128) shares of k, in
# fewer and more steps than a ring holds; tiles' remainders; more tiles than compute units
@pytest.mark.parametrize("m,n,k", [(33, 70, 32), (70, 33, 96), (100, 100, 160), (64, 64, 224), (65, 129, 288), (33, 65, 64), (40, 100, 192),
                                   (70, 70, 320), (90, 64, 448), (33, 33, 128), (50, 40, 256), (64, 100, 384), (33, 95, 640), (40, 40, 1152),
                                   (744, 2048, 1024), (2049, 1025, 96), (1100, 2100, 64)])
def test_float32_products_in_a_ring_of_slices(K, m, n, k):
    g = torch.Generator().manual_seed(m + n + k)
    a, w, c = torch.randn(m, k, generator=g), torch.randn(n, k, generator=g), torch.randn(m, n, generator=g)
    want = a.double() @ w.double().T
    out = torch.full((m, n), float("nan"), device="cuda:0")
    K.gemm(dev(a), dev(w), out)
    assert bool(((out.cpu().double() - want).abs() <= product_bound(a, w, k)).all())
    summed = dev(c)
    K.gemm(dev(a), dev(w), summed, accumulate=True)
    assert bool(((summed.cpu().double() - want - c).abs() <= product_bound(a, w, k) + 2.0 ** -24 * (want.abs() + c.abs() + 1)).all())


# more than a round of workgroups, K shorter than 256 (tiles) and from 256 on (slices), where the tiles' wide form is ahead of neither
@pytest.mark.parametrize("m,n,k", [(1100, 1100, 32), (1100, 1100, 224), (2049, 1025, 256), (600, 4100, 256), (1100, 2100, 288), (4100, 4097, 96)])
def test_float32_products_on_both_sides_of_short_k(K, m, n, k):
    test_float32_products_in_a_ring_of_slices(K, m, n, k)


@pytest.mark.parametrize("gate", ["silu", "gelu_tanh"])
@pytest.mark.parametrize("m,width,k", [(1, 3, 8), (4, 96, 128), (7, 4097, 68), (20, 40, 2304), (32, 8, 60), (33, 72, 64)])
def test_float32_gated_products(K, m, width, k, gate):
    """Against the activation of the very product's halves: what the one launch saves must not change the numbers."""
    g = torch.Generator().manual_seed(m + width + k)
    a, w = torch.randn(m, k, generator=g), torch.randn(2 * width, k, generator=g) / math.sqrt(k)
    both = a.double() @ w.double().T
    x, up = both[:, :width], both[:, width:]
    act = x * torch.sigmoid(x) if gate == "silu" else torch.nn.functional.gelu(x, approximate="tanh")
    out = torch.full((m, width), float("nan"), device="cuda:0")
    K.gemm_swiglu(dev(a), dev(w), out, gate)
    # both factors carry a product's error (the activation's slope is at most 1.13), and a few roundings of their own
    bound = product_bound(a, w, k)
    allowed = 1.13 * bound[:, :width] * up.abs() + bound[:, width:] * act.abs() + 2.0 ** -20 * (act * up).abs() + 1e-9
    assert bool(((out.cpu().double() - act * up).abs() <= allowed).all())


def test_float32_products_keep_infinities_to_their_rows(K):
    """Rows and weight rows beyond a tile's edge repeat the last one: nothing of them may reach another output."""
    for m, n in ((5, 9), (40, 70)):
        a, w = torch.ones(m, 64), torch.ones(n, 64)
        a[-1, 3], w[-1, 5] = float("inf"), float("nan")
        out = torch.empty(m, n, device="cuda:0")
        K.gemm(dev(a), dev(w), out)
        assert bool((out[:-1, :-1] == 64).all()) and bool(torch.isinf(out[-1, :-1]).all()) and bool(torch.isnan(out[:, -1]).all())


@pytest.mark.parametrize("n_heads,kv_heads,head_dim", [(2, 1, 32), (4, 2, 64), (3, 3, 96), (4, 1, 128), (2, 2, 192), (2, 1, 256)])
@pytest.mark.parametrize("window,chunk", [(0, 0), (70, 0), (0, 100)])
def test_float32_attention_rows_of_a_step(K, n_heads, kv_heads, head_dim, window, chunk):
    """Prompts whose rows share a workgroup, ends of sequences inside one, and one row a sequence; whatever stands behind a
    sequence's end (here NaN) stays out."""
    for pasts, news in (([0, 61, 5], [67, 3, 130]), ([0, 63, 64, 700], [1, 1, 1, 1])):
        lengths = [p + n for p, n in zip(pasts, news)]
        kp, vp, table, keys, values = make_cache(len(lengths), lengths, kv_heads, head_dim, torch.float32, seed=head_dim + window)
        for s, n in enumerate(lengths):
            if n % 64:
                kp[int(table[s, (n - 1) // 64]), :, n % 64:, :] = float("nan")
                vp[int(table[s, (n - 1) // 64]), :, :, n % 64:] = float("nan")
        positions = torch.tensor([p + t for p, n in zip(pasts, news) for t in range(n)], dtype=torch.int32)
        row_seq = torch.tensor([s for s, n in enumerate(news) for _ in range(n)], dtype=torch.int32)
        q = torch.randn(len(positions), n_heads * head_dim, generator=torch.Generator().manual_seed(1))
        out = torch.full(q.shape, float("nan"), device="cuda:0")
        starts = torch.tensor([0] + [sum(news[:i + 1]) for i in range(len(news))], dtype=torch.int32)
        layout = Layout(max(news) == 1, dev(starts), len(news), max(news), max(lengths) - 1)
        K.attention(dev(q), out, dev(kp), dev(vp), dev(table), dev(row_seq), dev(positions), n_heads, kv_heads, head_dim,
                    head_dim ** -0.5, window, layout=layout, chunk=chunk)
        got = out.cpu().double()
        for s in range(len(news)):
            rows = (row_seq == s).nonzero()[:, 0]
            at = positions[rows].long()
            for part in ([rows] if not chunk else [rows[at // chunk == c] for c in sorted(set((at // chunk).tolist()))]):
                first = int(positions[part[0]]) // chunk * chunk if chunk else 0
                want = attention_reference_rows(q[part], keys[s][first:], values[s][first:], positions[part].long() - first,
                                                n_heads, kv_heads, head_dim, head_dim ** -0.5, window)
                # probabilities carry the scores' error (sums of head_dim products of N(0, 1), divided by sqrt(head_dim)) and expf's
                assert float((got[part] - want).abs().max() / want.abs().max()) < 1e-5, (s, pasts)


def test_float32_attention_score_forms_and_ends(K):
    """Cap, slopes, temperature, sinks, gates and a factor, as the kernel for every size gives them (heads of 40 go there; zeros
    beyond 40 of 64 dimensions change no score)."""
    n_heads, kv_heads, lengths = 4, 2, [130, 3, 64]
    kp, vp, table, _, _ = make_cache(3, lengths, kv_heads, 64, torch.float32, seed=5)
    kp[..., 40:], vp[:, :, 40:] = 0.0, 0.0
    positions = torch.tensor([129, 2, 63], dtype=torch.int32)
    g = torch.Generator().manual_seed(2)
    q = torch.randn(3, n_heads, 64, generator=g)
    q[..., 40:] = 0.0
    gates = dev(torch.randn(3, n_heads, generator=g))
    more = dict(sinks=dev(torch.randn(n_heads, generator=g)), gates=gates, softcap=3.0, slopes=dev(torch.rand(n_heads, generator=g)),
                q_temp=(0.5, 16), out_scale=0.7)
    outs = []
    for size in (64, 40):
        out = torch.empty(3, n_heads * size, device="cuda:0")
        K.attention(dev(q[..., :size].reshape(3, -1).contiguous()), out, dev(kp[..., :size].contiguous()), dev(vp[:, :, :size].contiguous()),
                    dev(table), dev(torch.arange(3, dtype=torch.int32)), dev(positions), n_heads, kv_heads, size, 0.2, **more)
        outs.append(out.reshape(3, n_heads, size)[..., :40].double())
    assert float((outs[0] - outs[1]).abs().max() / outs[1].abs().max()) < 1e-5


@pytest.mark.parametrize("rows", [1, 12])
@pytest.mark.parametrize("blind", [(64, 128), (0, 64), (60, 200), (128, 197)])
def test_float32_attention_pages_of_keys_that_are_infinitely_far(K, rows, blind):
    """Keys with a score of minus infinity, a wave's whole first page of them, count for nothing beside keys that are seen."""
    n_heads, kv_heads, head_dim, length = 4, 2, 64, 300
    kp, vp, table, keys, values = make_cache(1, [length], kv_heads, head_dim, torch.float32, seed=rows)
    for t in range(*blind):
        kp[int(table[0, t // 64]), :, t % 64] = keys[0][t] = float("-inf")
    positions = torch.arange(length - rows, length, dtype=torch.int32)
    q = torch.rand(rows, n_heads * head_dim, generator=torch.Generator().manual_seed(2)) + 0.1
    out = torch.full(q.shape, float("nan"), device="cuda:0")
    layout = Layout(rows == 1, dev(torch.tensor([0, rows], dtype=torch.int32)), 1, rows, length - 1)
    K.attention(dev(q), out, dev(kp), dev(vp), dev(table), dev(torch.zeros(rows, dtype=torch.int32)), dev(positions), n_heads, kv_heads, head_dim,
                head_dim ** -0.5, layout=layout)
    want = attention_reference_rows(q, keys[0], values[0], positions.long(), n_heads, kv_heads, head_dim, head_dim ** -0.5, 0)
    assert float((out.cpu().double() - want).abs().max() / want.abs().max()) < 1e-5


# a page at most (prompts, a row a sequence, both ends of a page), four pages in enough rows and heads for a wave a row, and five
@pytest.mark.parametrize("n_heads,kv_heads,head_dim", [(4, 2, 32), (8, 4, 128), (6, 3, 160), (8, 2, 256)])
@pytest.mark.parametrize("pasts,news", [([0, 5, 63], [1, 1, 1]), ([0, 10], [64, 33]), ([0], [3]), ([0, 200, 100], [190, 56, 30]), ([0, 200], [190, 57]),
                                        ([50] * 150 + [255] * 20, [1] * 170)])
def test_float32_attention_of_few_pages(K, n_heads, kv_heads, head_dim, pasts, news):
    lengths = [p + n for p, n in zip(pasts, news)]
    kp, vp, table, keys, values = make_cache(len(lengths), lengths, kv_heads, head_dim, torch.float32, seed=head_dim)
    for s, n in enumerate(lengths):
        if n % 64:
            kp[int(table[s, (n - 1) // 64]), :, n % 64:, :] = float("nan")
            vp[int(table[s, (n - 1) // 64]), :, :, n % 64:] = float("nan")
    positions = torch.tensor([p + t for p, n in zip(pasts, news) for t in range(n)], dtype=torch.int32)
    row_seq = torch.tensor([s for s, n in enumerate(news) for _ in range(n)], dtype=torch.int32)
    q = torch.randn(len(positions), n_heads * head_dim, generator=torch.Generator().manual_seed(1))
    out = torch.full(q.shape, float("nan"), device="cuda:0")
    starts = torch.tensor([0] + [sum(news[:i + 1]) for i in range(len(news))], dtype=torch.int32)
    layout = Layout(max(news) == 1, dev(starts), len(news), max(news), max(lengths) - 1)
    K.attention(dev(q), out, dev(kp), dev(vp), dev(table), dev(row_seq), dev(positions), n_heads, kv_heads, head_dim, head_dim ** -0.5, layout=layout)
    got = out.cpu().double()
    for s in range(len(news)):
        rows = row_seq == s
        want = attention_reference_rows(q[rows], keys[s], values[s], positions[rows].long(), n_heads, kv_heads, head_dim, head_dim ** -0.5, 0)
        assert float((got[rows] - want).abs().max() / want.abs().max()) < 1e-5, s      # as in test_float32_attention_rows_of_a_step


# tiles of 16 columns: groups of 1, 3, 8 and 24 heads (columns of a row in two tiles), ends of sequences inside a tile, single rows
# between prompts, the last tile's columns that do not exist; the wave's 16 tokens before, at and behind a page's, window's or chunk's end
@pytest.mark.parametrize("n_heads,kv_heads,head_dim", [(16, 16, 32), (9, 3, 64), (16, 2, 128), (24, 1, 96), (8, 2, 256)])
@pytest.mark.parametrize("window,chunk", [(0, 0), (17, 0), (130, 0), (0, 48)])
def test_float32_attention_of_prompts_in_tiles(K, n_heads, kv_heads, head_dim, window, chunk):
    """Many columns of prompts; what a row does not see stays out although its neighbours in the tile see it: an infinite value of a
    later row's, NaN behind a sequence's end."""
    pasts, news = [0, 15, 0, 64, 130], [16, 1, 190, 3, 77]
    lengths = [p + n for p, n in zip(pasts, news)]
    kp, vp, table, keys, values = make_cache(len(lengths), lengths, kv_heads, head_dim, torch.float32, seed=head_dim + window)
    for s, n in enumerate(lengths):
        if n % 64:
            kp[int(table[s, (n - 1) // 64]), :, n % 64:, :] = float("nan")
            vp[int(table[s, (n - 1) // 64]), :, :, n % 64:] = float("nan")
    far, dim = 100, head_dim - 3       # the third sequence's row 100 holds an infinite value
    vp[int(table[2, far // 64]), :, dim, far % 64] = values[2][far][:, dim] = float("inf")
    positions = torch.tensor([p + t for p, n in zip(pasts, news) for t in range(n)], dtype=torch.int32)
    row_seq = torch.tensor([s for s, n in enumerate(news) for _ in range(n)], dtype=torch.int32)
    q = torch.randn(len(positions), n_heads * head_dim, generator=torch.Generator().manual_seed(1))
    out = torch.full(q.shape, float("nan"), device="cuda:0")
    starts = torch.tensor([0] + [sum(news[:i + 1]) for i in range(len(news))], dtype=torch.int32)
    layout = Layout(False, dev(starts), len(news), max(news), max(lengths) - 1)
    assert len(positions) >= 32 * len(news) and len(positions) * n_heads > 2048
    K.attention(dev(q), out, dev(kp), dev(vp), dev(table), dev(row_seq), dev(positions), n_heads, kv_heads, head_dim, head_dim ** -0.5, window,
                layout=layout, chunk=chunk)
    got = out.cpu().double().reshape(len(positions), n_heads, head_dim)
    finite = [v.clone() for v in values]
    finite[2][far][:, dim] = 0.0
    for s in range(len(news)):
        rows = (row_seq == s).nonzero()[:, 0]
        at = positions[rows].long()
        first = at // chunk * chunk if chunk else (at - window + 1 if window else at * 0)
        for part in ([rows] if not chunk else [rows[at // chunk == c] for c in sorted(set((at // chunk).tolist()))]):
            lead = int(positions[part[0]]) // chunk * chunk if chunk else 0
            want = attention_reference_rows(q[part], keys[s][lead:], finite[s][lead:], positions[part].long() - lead,
                                            n_heads, kv_heads, head_dim, head_dim ** -0.5, window).reshape(len(part), n_heads, head_dim)
            mine = got[part].clone()
            if s == 2:
                sees = ((positions[part].long() >= far) & (first[torch.isin(rows, part)] <= far))
                assert bool((mine[sees][:, :, dim] == float("inf")).all())
                mine[sees, :, dim], want[sees, :, dim] = 0.0, 0.0
            # as in test_float32_attention_rows_of_a_step
            assert float((mine - want).abs().max() / want.abs().max()) < 1e-5, s


def test_float32_attention_of_prompts_in_tiles_score_forms_and_ends(K):
    """Cap, slopes, temperature, sinks, gates and a factor, as the kernel for every size gives them."""
    n_heads, kv_heads, length = 12, 4, 200
    kp, vp, table, _, _ = make_cache(1, [length], kv_heads, 64, torch.float32, seed=5)
    kp[..., 40:], vp[:, :, 40:] = 0.0, 0.0
    g = torch.Generator().manual_seed(2)
    q = torch.randn(length, n_heads, 64, generator=g)
    q[..., 40:] = 0.0
    more = dict(sinks=dev(torch.randn(n_heads, generator=g)), gates=dev(torch.randn(length, n_heads, generator=g)), softcap=3.0,
                slopes=dev(torch.rand(n_heads, generator=g)), q_temp=(0.5, 16), out_scale=0.7)
    outs = []
    for size in (64, 40):
        out = torch.empty(length, n_heads * size, device="cuda:0")
        K.attention(dev(q[..., :size].reshape(length, -1).contiguous()), out, dev(kp[..., :size].contiguous()), dev(vp[:, :, :size].contiguous()),
                    dev(table), dev(torch.zeros(length, dtype=torch.int32)), dev(torch.arange(length, dtype=torch.int32)), n_heads, kv_heads,
                    size, 0.2, **more)
        outs.append(out.reshape(length, n_heads, size)[..., :40].double())
    assert float((outs[0] - outs[1]).abs().max() / outs[1].abs().max()) < 1e-5


@pytest.mark.parametrize("pasts,tiled", [([0] + [900] * 6, False), ([0] * 7, True)])
def test_float32_attention_of_a_prompt_beside_decoding_rows(K, pasts, tiled):
    """A step that says how its rows group into sequences: rows behind many keys keep the step out of the tiles, rows behind few do not;
    the results are the same sums either way."""
    import ctypes
    from types import SimpleNamespace
    n_heads, kv_heads, head_dim, news = 16, 8, 128, [300] + [1] * 6
    lengths = [p + n for p, n in zip(pasts, news)]
    kp, vp, table, keys, values = make_cache(len(lengths), lengths, kv_heads, head_dim, torch.float32, seed=3)
    starts = [sum(news[:i]) for i in range(len(news) + 1)]
    assert bool(K.lib.bh_attention_f32_tiles(starts[-1], len(news), n_heads, kv_heads, head_dim, 0, (ctypes.c_int32 * len(starts))(*starts),
                                             (ctypes.c_int32 * len(pasts))(*pasts))) == tiled
    positions = torch.tensor([p + t for p, n in zip(pasts, news) for t in range(n)], dtype=torch.int32)
    row_seq = torch.tensor([s for s, n in enumerate(news) for _ in range(n)], dtype=torch.int32)
    layout = SimpleNamespace(is_decode=False, seq_start=dev(torch.tensor(starts, dtype=torch.int32)), n_seqs=len(news), max_rows_per_seq=max(news),
                             max_position=max(lengths) - 1, host_seq_start=starts, host_seq_past=pasts)
    q = torch.randn(len(positions), n_heads * head_dim, generator=torch.Generator().manual_seed(1))
    out = torch.full(q.shape, float("nan"), device="cuda:0")
    K.attention(dev(q), out, dev(kp), dev(vp), dev(table), dev(row_seq), dev(positions), n_heads, kv_heads, head_dim, head_dim ** -0.5,
                layout=layout)
    for s in range(len(news)):
        rows = slice(starts[s], starts[s + 1])
        want = attention_reference_rows(q[rows], keys[s], values[s], positions[rows].long(), n_heads, kv_heads, head_dim, head_dim ** -0.5, 0)
        # as in test_float32_attention_rows_of_a_step
        assert float((out[rows].cpu().double() - want).abs().max() / want.abs().max()) < 1e-5, s
