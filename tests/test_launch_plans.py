"""The kernel library's launch decisions that are plain host arithmetic: asked of the built library without a GPU
(`KernelSizes`), at the compute-unit count it assumes there (256)."""

import pytest
import torch

from beholdd.kernels import KernelSizes


@pytest.fixture(scope="module")
def sizes():
    import ctypes
    library = KernelSizes(verbose_build=False)
    i = ctypes.c_int
    library.lib.bh_attention_bf16_splits.argtypes, library.lib.bh_attention_bf16_splits.restype = [i] * 5, i
    library.lib.bh_gemm_bf16_norm_blocks.argtypes, library.lib.bh_gemm_bf16_norm_blocks.restype = [i] * 5, i
    return library


def workgroups(sizes, sequences, context, heads=32, kv_heads=8):
    splits = sizes.lib.bh_attention_bf16_splits(sequences, 1, heads, kv_heads, context - 1)
    return splits, sequences * kv_heads * splits


def test_key_splits_fill_whole_rounds_of_workgroups(sizes):
    """A decode step's attention runs in rounds of one workgroup per compute unit: the split count never leaves a
    second round of a few workgroups that are sized for one round (288 to 384 of them for 9 to 14 sequences before)."""
    assert workgroups(sizes, 8, 8192) == (4, 256)
    assert workgroups(sizes, 1, 8192) == (32, 256)
    assert workgroups(sizes, 16, 8192) == (2, 256)
    assert workgroups(sizes, 32, 8192) == (1, 256)
    assert workgroups(sizes, 12, 8192) == (5, 480)
    assert workgroups(sizes, 6, 8192) == (5, 240)
    for sequences in range(1, 33):
        splits, count = workgroups(sizes, sequences, 8192)
        rounds = -(-count // 256)
        assert count > 0.75 * rounds * 256, (sequences, splits, count)      # no round of a few workgroups behind full ones
        assert splits <= 128 // 4                                           # every wave of a workgroup has a page
    # more workgroups than compute units: three splits just above one per compute unit, two just above two, else none
    assert [workgroups(sizes, n, 8192)[0] for n in (33, 40, 44, 48, 56, 64, 68, 72, 80, 128)] == [3, 3, 3, 1, 1, 1, 2, 2, 1, 1]
    # short caches are not split (fewer than eight pages), and a split never has fewer than four pages
    assert workgroups(sizes, 8, 448)[0] == 1 and workgroups(sizes, 8, 640)[0] == 2 and workgroups(sizes, 1, 1024)[0] == 4


def test_the_norm_that_rides_counts_the_workgroups_of_wider_spans(sizes):
    """Products of up to 32 rows whose blocks of 16 weight rows number between one and two per compute unit run with
    workgroups of 20 or 24 rows; a norm behind such a product gets one partial sum per workgroup."""
    blocks = lambda m, n, k: sizes.lib.bh_gemm_bf16_norm_blocks(m, n, k, 1, 0)
    assert blocks(8, 4096, 4096) == 256            # one block of 16 rows per compute unit
    assert blocks(8, 5120, 5120) == 256            # 320 blocks: spans of 20 rows
    assert blocks(32, 6144, 4096) == 256           # 384 blocks: spans of 24 rows
    assert blocks(8, 7168, 5120) == 448            # 28 rows could lie in three blocks: left to the blocks of 16
    assert blocks(8, 8192, 4096) == 512 and blocks(8, 2560, 4096) == 160


def test_prepared_rows_reach_no_product_that_does_not_scale(sizes):
    """From 129 rows on the kernel for many rows takes a gated product, whose output it may write in blocks but whose sums it does
    not scale: it takes no prepared rows; products take them where K goes in parts, whose finishing kernel scales."""
    takes, writes, scratch = sizes.lib.bh_gemm_bf16_takes_norm, sizes.lib.bh_gemm_bf16_writes_blocked, sizes.lib.bh_gemm_bf16_scratch
    for m in (129, 160, 200, 256, 300, 1000):
        for k in (64, 512, 1024, 2048, 4096, 9216):
            for n in (128, 512, 1024, 3072, 9216, 27648):
                if takes(m, n, k, 1, 1) and writes(m, n, k, 1, 1):
                    assert sizes.lib.bh_gemm_bf16_plan(m, n, k, 1, 1) < 0 and scratch(m, n, k, 1, 1) > 0, (m, n, k)
                if sizes.lib.bh_gemm_bf16_reads_blocked(m, n, k, 1, 0) and takes(m, n, k, 1, 0):
                    assert scratch(m, n, k, 1, 0) > 0, (m, n, k)


def test_a_launch_that_writes_rows_refuses_an_output_in_blocks(sizes):
    """The tiles know rows only: the entry for all products refuses what would reach them with an output in blocks, prepared rows or
    activations in rows, before anything is launched."""
    if torch.cuda.is_available():
        pytest.skip("made-up addresses: only where nothing can be launched")
    at = 1 << 20
    for ahead, why in ((at, "cannot take prepared norm rows"), (None, "does not write these blocks")):
        status = sizes.lib.bh_gemm_bf16(at, at, at, 1, 0, 200, 3072, 1024, 1, 1, ahead, 16 if ahead else 0, 1e-6 if ahead else 0.0,
                                        None, 0, None, None, None, 0, 16, 0, None)
        assert status != 0 and why in sizes.lib.bh_last_error().decode(), ahead


def float32_tiles(sizes, lengths, pasts, heads, kv_heads, head_dim, window=0):
    import ctypes
    starts = [sum(lengths[:i]) for i in range(len(lengths) + 1)]
    return bool(sizes.lib.bh_attention_f32_tiles(starts[-1], len(lengths), heads, kv_heads, head_dim, window,
                                                 (ctypes.c_int32 * len(starts))(*starts), (ctypes.c_int32 * len(pasts))(*pasts)))


def test_float32_prompts_go_in_tiles_unless_short_rows_look_far(sizes):
    """A tile of 16 columns walks its sequences one after another: prompts go in tiles, and so do rows that share a sequence behind any
    number of keys, but not decoding rows one behind the other in a tile behind many keys."""
    alone = lambda *lengths: (list(lengths), [0] * len(lengths))
    for lengths, pasts in (alone(2048), alone(300, 186, 200, 58), alone(700, 300), alone(*[120] * 8), ([64] * 8, [1000] * 8), ([64] * 8, [8000] * 8)):
        for heads, kv_heads, head_dim in ((8, 4, 128), (16, 2, 128), (32, 8, 128), (8, 2, 256), (16, 16, 64)):
            assert float32_tiles(sizes, lengths, pasts, heads, kv_heads, head_dim), (lengths, heads, kv_heads, head_dim)
    # 8 rows of a sequence each in a tile, 2, 4 and 16
    for heads, kv_heads, head_dim in ((8, 4, 128), (16, 2, 128), (32, 8, 128), (16, 16, 64)):
        assert not float32_tiles(sizes, [500] + [1] * 14, [0] + [8000] * 14, heads, kv_heads, head_dim)
        assert not float32_tiles(sizes, [512, 1], [0, 8000], heads, kv_heads, head_dim)
    # a window or a chunk bounds what a row sees
    assert float32_tiles(sizes, [500] + [1] * 14, [0] + [8000] * 14, 32, 8, 128, 64)
    assert float32_tiles(sizes, [500] + [1] * 14, [0] + [8000] * 14, 32, 8, 128, -64)
    assert not float32_tiles(sizes, [2000] + [1] * 60, [0] + [4000] * 60, 8, 4, 128)
    assert float32_tiles(sizes, [2000] + [1] * 60, [0] + [500] * 60, 8, 4, 128)
    assert float32_tiles(sizes, [2000] + [1] * 60, [0] + [4000] * 60, 32, 8, 128)
    # few rows a sequence, or few rows and heads: never
    assert not float32_tiles(sizes, [31] * 8, [0] * 8, 32, 8, 128) and not float32_tiles(sizes, [64], [0], 16, 8, 128)


TILES = ["128x128", "128x128 in halves", "256x128", "256x192", "256x256"]


def many_rows_plan(sizes, m, n, k, output):
    """(tile, parts of K) of a product of many rows, or None; `output`: "float32", "gated" or "bfloat16"."""
    plan = sizes.lib.bh_gemm_bf16_plan(m, n, k, 1, ["float32", "gated", "bfloat16"].index(output))
    return (TILES[plan // 16], plan % 16) if plan >= 0 else None


def test_products_of_many_rows_take_the_tiles_that_were_measured_fastest(sizes):
    """Sizes at which the choice matters: what is chosen / the next best of another kind, us, the launches behind them included."""
    plan = lambda *size: many_rows_plan(sizes, *size)
    assert plan(768, 4096, 12288, "float32") == ("256x256", 4)              # 88 / 105 on 128 x 128 in 4 parts
    assert plan(1500, 4096, 12288, "float32") == ("256x256", 2)             # 143 / 159 on 256 x 128
    assert plan(1500, 4096, 4096, "float32") == ("256x128", 1)              # 70 / 78 on 128 x 128 in 2 parts
    assert plan(1000, 5120, 5120, "float32") == ("256x192", 2)              # 72 / 78 on 256 x 128, 98 on 128 x 128 in 2
    assert plan(1300, 2048, 2048, "bfloat16") == ("128x128", 1)             # 23 / 27 in 2 parts
    assert plan(2100, 1024, 1024, "bfloat16") == ("128x128", 1)             # 14 / 19 on 256 x 128
    assert plan(1800, 3072, 2048, "bfloat16")[0] in ("128x128", "256x128")  # 32 / 40 in halves
    assert plan(640, 17408, 5120, "gated") == ("256x256", 1)                # 231 / 253 on 128 x 128
    assert plan(256, 12288, 4096, "gated") == ("256x128", 1)                # 66 / 78 on 128 x 128
    # gated products of few tiles: the whole tiles with K in parts
    assert plan(256, 1024, 4096, "gated") is None and plan(129, 2048, 2048, "gated") is None and plan(512, 768, 2048, "gated") is None
    assert plan(400, 2048, 2048, "gated") is not None and plan(129, 6912, 2560, "gated") is not None
    # slices of k that make no equal parts, or none fine enough: the whole tiles again, whatever the product writes
    for size in ((278, 960, 4544), (478, 768, 7232), (148, 2816, 4544), (264, 640, 1984), (675, 960, 3904), (862, 1344, 7744)):
        assert plan(*size, "float32") is None and plan(*size, "bfloat16") is None, size
    assert plan(1140, 1280, 2752, "float32") is not None
    assert plan(128, 4096, 4096, "float32") is None and plan(256, 4096, 512, "float32") is None      # for the slices; the tiles


def test_sums_left_in_parts_are_in_the_byte_plan(sizes):
    """`gemm_bare` hands out the sums of K's parts, also where the product itself adds up two halves of k and needs no scratch memory:
    what a projection that may be left in parts is planned with covers them, beside its regrouped activations."""
    from beholdd.kernels.library import BlockedRows
    halves = 0
    for width, outputs in ((1024, 2048), (2048, 4096), (2560, 3584), (4096, 2048), (4096, 6144), (4096, 8192), (5120, 7168)):
        for m in list(range(129, 1100, 23)) + [1500, 2048, 3000]:
            parts = sizes.lib.bh_gemm_bf16_bare_parts(m, outputs, width, 1)
            sums = parts * m * outputs * 4
            halves += parts == 2 and sizes.lib.bh_gemm_bf16_scratch(m, outputs, width, 1, 0) < sums
            planned = sizes.gemm_working_bytes(m, outputs, width, 2, bare=True)
            assert planned >= sums + 2 * BlockedRows.padded_rows(m, 16) * width * 2, (m, outputs, width, parts)
    assert halves > 0      # sizes among them that scratch memory alone does not cover


def test_experts_tiles_of_pairs_follow_the_rounds(sizes):
    """Pairs of a tile of the routed experts' products: where both widths were timed (32 experts unless said)."""
    gate_up = lambda pairs, width, ff, experts=32: sizes.lib.bh_experts_many_tile(pairs * experts, experts, width, ff, 1)
    down = lambda pairs, width, ff, experts=32: sizes.lib.bh_experts_many_tile(pairs * experts, experts, ff, width, 0)
    assert [gate_up(n, 1024, 384) for n in (16, 48, 56, 128)] == [64] * 4 and gate_up(192, 1024, 384) == 128
    assert [gate_up(n, 2048, 768) for n in (16, 48, 56)] == [64] * 3 and [gate_up(n, 2048, 768) for n in (64, 96, 192)] == [128] * 3
    assert down(48, 2048, 768) == 64 and down(56, 2048, 768) == 128
    assert [gate_up(n, 4096, 1536) for n in (16, 96, 256)] == [128] * 3
    assert gate_up(56, 2048, 1408, 8) == 64 and gate_up(64, 2048, 1408, 8) == 128 and gate_up(40, 2048, 768, 128) == 64
