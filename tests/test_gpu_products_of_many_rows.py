"""Products of more than 128 rows of packed weights on every tile they are compiled for, at the tiles' edges, against float64."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    from beholdd.kernels import HipKernels
    return HipKernels()


def rel(got, want):
    got = got.double().cpu() if got.dtype != torch.float64 else got.cpu()
    return float((got - want).abs().max() / want.abs().max())


# rows, weight rows and k one beyond and one short of whole tiles, of whole steps in the ring (64 k are two), of parts of K; which tiles
# they run on is an estimate's choice (`test_every_tile_and_cut_of_the_products_of_many_rows` holds sizes to theirs)
SIZES = [(129, 1024, 1024), (129, 1040, 1088), (256, 1024, 1152), (257, 128, 128), (257, 144, 192), (383, 1008, 320),
         (2049, 2064, 1088), (2049, 2032, 1152), (2048, 2048, 2048), (2096, 3088, 512), (2047, 4096, 640), (1025, 4112, 256),
         (2049, 6128, 256), (251, 5120, 2048), (140, 7168, 1280), (700, 6160, 2048), (8193, 4080, 128)]


@pytest.mark.parametrize("m,n,k", SIZES)
def test_products_of_many_rows(K, m, n, k):
    """float32 with and without accumulation, bfloat16 and gated, from activations whose buffer holds NaN behind the last row; the
    bounds are those of a sum of k float32 products and of one bfloat16 rounding."""
    from beholdd.kernels.library import BlockedRows
    g = torch.Generator(device="cuda:0").manual_seed(m + n + k)
    a = torch.randn(m, k, generator=g, device="cuda:0").to(torch.bfloat16)
    w = (torch.randn(2 * n, k, generator=g, device="cuda:0") * 0.05).to(torch.bfloat16)
    plain, both = K.pack_weight(w[:n].contiguous()), K.pack_weight(w)
    in_blocks = BlockedRows(torch.full((BlockedRows.padded_rows(m, 16) * k,), float("nan"), dtype=torch.bfloat16, device="cuda:0"), m, k)
    K.to_blocked(a, in_blocks)
    want, up = (a.double() @ w[:n].double().t()).cpu(), (a.double() @ w[n:].double().t()).cpu()
    bound = 4 * math.sqrt(k) * 2.0 ** -24
    for x in (in_blocks, a):
        out = torch.full((m, n), float("nan"), dtype=torch.float32, device="cuda:0")
        K.gemm(x, plain, out)
        assert rel(out, want) < bound
    base = torch.randn(m, n, generator=g, device="cuda:0")
    total = base.clone()
    K.gemm(in_blocks, plain, total, accumulate=True)
    assert rel(total, want + base.double().cpu()) < bound
    rounded = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda:0")
    K.gemm(in_blocks, plain, rounded)
    assert rel(rounded, want) < 4e-3
    gated = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda:0")
    K.gemm_swiglu(in_blocks, both, gated)
    assert rel(gated, want / (1 + torch.exp(-want)) * up) < 6e-3
    if n % 32 == 0:
        blocked = K.new_rows(m, n, torch.bfloat16, n, False)
        K.gemm_swiglu(in_blocks, both, blocked)
        assert torch.equal(K.from_blocked(blocked) if isinstance(blocked, BlockedRows) else blocked, gated)


@pytest.mark.parametrize("m,n,k", [(251, 5120, 2048), (129, 1024, 1024), (2048, 2048, 2048), (300, 4096, 1088)])
def test_products_of_many_rows_and_the_norm_behind_them(K, m, n, k):
    """`gemm(..., then_norm=)`: the residual as without the norm bit for bit, and its norm within a bfloat16 rounding."""
    from beholdd.kernels.library import BlockedRows
    from beholdd.parts.base import NormRequest, ProductReader
    g = torch.Generator(device="cuda:0").manual_seed(m + n)
    a = torch.randn(m, k, generator=g, device="cuda:0").to(torch.bfloat16)
    packed = K.pack_weight((torch.randn(n, k, generator=g, device="cuda:0") * 0.05).to(torch.bfloat16))
    base, weight = torch.randn(m, n, generator=g, device="cuda:0"), 1 + 0.3 * torch.randn(n, generator=g, device="cuda:0")
    plain, residual = base.clone(), base.clone()
    K.gemm(a, packed, plain, accumulate=True)
    normed = K.gemm(a, packed, residual, accumulate=True, then_norm=NormRequest(weight, 1e-5, ProductReader(n)))
    assert torch.equal(plain, residual)
    got = residual.double()
    want = got / torch.sqrt((got ** 2).mean(-1, keepdim=True) + 1e-5) * weight.double()
    assert rel(K.from_blocked(normed) if isinstance(normed, BlockedRows) else normed, want.cpu()) < 4e-3


TILES = ["128x128", "128x128 in halves", "256x128", "256x192", "256x256"]


def plan(K, m, n, k, output):
    """(tile, parts of K) on the kernel for many rows; `output`: float32, gated or bfloat16."""
    code = int(K.lib.bh_gemm_bf16_plan(m, n, k, 1, ["float32", "gated", "bfloat16"].index(output)))
    return (TILES[code // 16], code % 16) if code >= 0 else None


# every tile with K whole and in parts, where it is compiled for that output, at sizes that no tile divides; the plan is asserted, so that
# another estimate cannot empty this
@pytest.mark.parametrize("output,tile,parts,m,n,k", [
    ("float32", "128x128", 1, 257, 144, 128), ("float32", "128x128", 2, 257, 144, 512), ("float32", "128x128 in halves", 1, 257, 8208, 3072),
    ("float32", "256x128", 1, 385, 8208, 128), ("float32", "256x128", 4, 129, 4112, 2048), ("float32", "256x192", 1, 900, 8208, 128),
    ("float32", "256x192", 4, 129, 8208, 4096), ("float32", "256x256", 1, 1300, 8208, 128), ("float32", "256x256", 5, 257, 6160, 5120),
    ("gated", "128x128", 1, 257, 144, 128), ("gated", "128x128 in halves", 1, 129, 5136, 3072), ("gated", "256x128", 1, 257, 6160, 128),
    ("gated", "256x192", 1, 385, 8208, 128), ("gated", "256x256", 1, 257, 12304, 128),
    ("bfloat16", "128x128", 1, 257, 144, 128), ("bfloat16", "128x128", 4, 257, 144, 1024), ("bfloat16", "128x128 in halves", 1, 520, 4112, 3072),
    ("bfloat16", "256x128", 1, 385, 8208, 128), ("bfloat16", "256x128", 4, 129, 4112, 2048), ("bfloat16", "256x192", 1, 900, 8208, 128),
    ("bfloat16", "256x192", 4, 129, 8208, 2048), ("bfloat16", "256x256", 1, 1300, 8208, 128), ("bfloat16", "256x256", 8, 129, 6160, 6144)])
def test_every_tile_and_cut_of_the_products_of_many_rows(K, output, tile, parts, m, n, k):
    """From activations whose buffer holds NaN behind the last row; the bounds are those of `test_products_of_many_rows`."""
    from beholdd.kernels.library import BlockedRows
    assert plan(K, m, n, k, output) == (tile, parts)
    g = torch.Generator(device="cuda:0").manual_seed(m + n + k)
    a = torch.randn(m, k, generator=g, device="cuda:0").to(torch.bfloat16)
    w = (torch.randn((2 if output == "gated" else 1) * n, k, generator=g, device="cuda:0") * 0.05).to(torch.bfloat16)
    in_blocks = BlockedRows(torch.full((BlockedRows.padded_rows(m, 16) * k,), float("nan"), dtype=torch.bfloat16, device="cuda:0"), m, k)
    K.to_blocked(a, in_blocks)
    want = a.double() @ w[:n].double().t()
    if output == "gated":
        want = want / (1 + torch.exp(-want)) * (a.double() @ w[n:].double().t())
        out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda:0")
        K.gemm_swiglu(in_blocks, K.pack_weight(w), out)
        assert rel(out, want.cpu()) < 6e-3
        return
    base = torch.randn(m, n, generator=g, device="cuda:0")
    out = base.clone() if output == "float32" else torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda:0")
    K.gemm(in_blocks, K.pack_weight(w), out, accumulate=output == "float32")
    if output == "float32":
        assert rel(out, (want + base.double()).cpu()) < 4 * math.sqrt(k) * 2.0 ** -24
    else:
        assert rel(out, want.cpu()) < 4e-3


# the kernel that adds up the parts and finishes the norm, with one, two, four and eight rows a block, for up to two, four and eight parts
@pytest.mark.parametrize("m,n,k,parts", [(257, 192, 512, 2), (257, 192, 768, 3), (333, 4096, 12288, 4), (257, 192, 1536, 6),
                                         (520, 192, 512, 2), (520, 192, 768, 3), (520, 192, 1536, 6), (2049, 192, 512, 2), (2049, 192, 768, 3),
                                         (2049, 128, 1536, 6), (2056, 2048, 6144, 3), (4097, 192, 768, 2), (4097, 192, 1536, 3), (4097, 192, 5120, 5)])
@pytest.mark.parametrize("blocked", [False, True])
def test_norm_finished_from_parts_with_every_number_of_rows_a_block(K, m, n, k, parts, blocked):
    """The residual as without the norm bit for bit; the norm within a bfloat16 rounding of float64's, in rows and in its reader's blocks."""
    from beholdd.kernels.library import BlockedRows
    from beholdd.parts.base import NormRequest, ProductReader
    assert plan(K, m, n, k, "float32")[1] == parts
    g = torch.Generator(device="cuda:0").manual_seed(m + k)
    a = torch.randn(m, k, generator=g, device="cuda:0").to(torch.bfloat16)
    packed = K.pack_weight((torch.randn(n, k, generator=g, device="cuda:0") / k ** 0.5).to(torch.bfloat16))
    base, weight = torch.randn(m, n, generator=g, device="cuda:0"), 1 + 0.3 * torch.randn(n, generator=g, device="cuda:0")
    without, residual = base.clone(), base.clone()
    K.gemm(a, packed, without, accumulate=True)
    normed = K.gemm(a, packed, residual, accumulate=True, then_norm=NormRequest(weight, 1e-5, ProductReader(4096) if blocked else None))
    assert torch.equal(without, residual) and isinstance(normed, BlockedRows) == blocked
    got = residual.double()
    want = got / torch.sqrt((got ** 2).mean(-1, keepdim=True) + 1e-5) * weight.double()
    assert rel(K.from_blocked(normed) if blocked else normed, want.cpu()) < 4e-3


# slices of k that divide into no parts that are alike: the whole tiles cut them unevenly; with the norm behind and in front of them
@pytest.mark.parametrize("m,n,k", [(148, 2816, 4544), (264, 640, 1984), (291, 832, 2752), (500, 768, 7232), (675, 960, 3904), (862, 1344, 7744)])
def test_products_whose_slices_make_no_equal_parts(K, m, n, k):
    from beholdd.kernels.library import BlockedRows
    from beholdd.parts.base import NormRequest, ProductReader
    assert plan(K, m, n, k, "float32") is None and plan(K, m, n, k, "bfloat16") is None and K.lib.bh_gemm_bf16_scratch(m, n, k, 1, 0) > 0
    g = torch.Generator(device="cuda:0").manual_seed(m + n + k)
    a = torch.randn(m, k, generator=g, device="cuda:0").to(torch.bfloat16)
    w = (torch.randn(n, k, generator=g, device="cuda:0") / k ** 0.5).to(torch.bfloat16)
    next_w = (torch.randn(2 * 1024, n, generator=g, device="cuda:0") / n ** 0.5).to(torch.bfloat16)
    packed, base, weight = K.pack_weight(w), torch.randn(m, n, generator=g, device="cuda:0"), 1 + 0.3 * torch.randn(n, generator=g, device="cuda:0")
    want = a.double() @ w.double().t()
    for x in (a, K.to_blocked(a)):
        out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda:0")
        K.gemm(x, packed, out)
        assert rel(out, want.cpu()) < 4e-3
    assert K.gemm_bare(a, packed) is None
    residual = base.clone()
    prepared = K.gemm(a, packed, residual, accumulate=True, then_norm=NormRequest(weight, 1e-5, ProductReader(1024, True)))
    residual64 = want + base.double()
    assert rel(residual, residual64.cpu()) < 4 * math.sqrt(k) * 2.0 ** -24
    if prepared is None:
        prepared = K.new_rows(m, n, torch.bfloat16, 1024, True)
        K.rmsnorm(residual, weight, 1e-5, prepared)
    gated = K.new_rows(m, 1024, torch.bfloat16, 512)
    K.gemm_swiglu(prepared, K.pack_weight(next_w), gated)
    normed = residual64 / torch.sqrt((residual64 ** 2).mean(-1, keepdim=True) + 1e-5) * weight.double()
    both = normed @ next_w.double().t()
    # the norm's rows and the gated output are rounded to 8 bits, rows that wait for their factor as well
    assert rel(K.from_blocked(gated) if isinstance(gated, BlockedRows) else gated, (both[:, :1024] / (1 + torch.exp(-both[:, :1024])) * both[:, 1024:]).cpu()) < 1.2e-2


# few rows (blocks of 8 and of 16, one and two blocks of rows), 33 to 128 rows and spans of 24 weight rows (two launches), many rows on
# every kind of tile, K in parts (two launches); rows and columns that no tile divides
@pytest.mark.parametrize("m,n,k", [(1, 96, 128), (8, 544, 192), (9, 4096, 256), (16, 160, 64), (17, 96, 1088), (32, 12288, 128), (16, 6144, 128),
                                   (40, 512, 256), (129, 1056, 1024), (257, 1600, 1088), (300, 17408, 256), (1000, 4128, 2048),
                                   (2100, 6144, 256), (4100, 8224, 128), (256, 2048, 4096)])
def test_products_squared_behind_a_relu(K, m, n, k):
    g = torch.Generator().manual_seed(m + n + k)
    a, w = torch.randn(m, k, generator=g).bfloat16(), (torch.randn(n, k, generator=g) / k ** 0.5).bfloat16()
    packed, a_rows = K.pack_weight(w.cuda()), a.cuda()
    exact = (a_rows.double() @ w.cuda().double().T).clamp(min=0.0)
    # float32 sums of k products, squared; the result rounded to 8 bits
    error = 2.0 ** -23 * k ** 0.5 * 4.0
    bound = 2.0 ** -8 * exact ** 2 + 2 * exact * error + error ** 2 + 1e-30
    for block_rows in (0, 8, 16):
        out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda:0") if not block_rows else K.to_blocked(
            torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda:0"), block_rows=block_rows)
        taken = K.gemm_relu_squared(a_rows, packed, out)
        kind = int(K.lib.bh_gemm_bf16_squares(m, n, k))
        assert taken == (kind == 2 or (kind == 1 and block_rows != 8))
        assert kind == (0 if (m, n) in ((16, 6144), (40, 512), (129, 1056), (256, 2048)) else 2 if m <= 32 else 1)
        if taken:
            got = (K.from_blocked(out) if block_rows else out).double()
            assert bool(((got - exact ** 2).abs() <= bound).all()), block_rows


# gated products whose K the whole tiles cut into parts: the finishing kernel writes rows or the blocks that a product of many rows reads
@pytest.mark.parametrize("m,inter,k", [(129, 1024, 1024), (200, 1056, 4096), (256, 2048, 2048), (400, 768, 2048)])
def test_gated_products_of_few_tiles(K, m, inter, k):
    from beholdd.kernels.library import BlockedRows
    assert int(K.lib.bh_gemm_bf16_plan(m, inter, k, 1, 1)) < 0 and K.lib.bh_gemm_bf16_scratch(m, inter, k, 1, 1) > 0
    g = torch.Generator(device="cuda:0").manual_seed(m + inter)
    a = torch.randn(m, k, generator=g, device="cuda:0").to(torch.bfloat16)
    w = (torch.randn(2 * inter, k, generator=g, device="cuda:0") / k ** 0.5).to(torch.bfloat16)
    gate, up = (a.double() @ half.double().t() for half in (w[:inter], w[inter:]))
    packed, rows = K.pack_weight(w), torch.full((m, inter), float("nan"), dtype=torch.bfloat16, device="cuda:0")
    K.gemm_swiglu(a, packed, rows)
    assert rel(rows, (gate / (1 + torch.exp(-gate)) * up).cpu()) < 6e-3
    blocks = K.to_blocked(torch.full((m, inter), float("nan"), dtype=torch.bfloat16, device="cuda:0"))
    K.gemm_swiglu(K.to_blocked(a), packed, blocks)
    assert isinstance(blocks, BlockedRows) and torch.equal(K.from_blocked(blocks), rows)


# hidden and attention widths whose output projection prepares the norm behind it (K below 1,024: tiles; more than 8,192 outputs: parts
# of K and their finishing kernel) in front of a gated product of the kernel for many rows
@pytest.mark.parametrize("hidden,attention,inter", [(1024, 512, 3072), (1024, 512, 1024), (9216, 9216, 2048)])
@pytest.mark.parametrize("m", [129, 200, 256])
def test_norms_between_products_of_129_to_256_rows(K, m, hidden, attention, inter):
    """o -> norm -> gate and up into the down product's blocks -> down, with and without the norm's reader named, against float64."""
    from beholdd.parts.base import NormRequest, ProductReader
    g = torch.Generator(device="cuda:0").manual_seed(m + hidden)
    normal = lambda *shape: torch.randn(*shape, generator=g, device="cuda:0")
    attended = normal(m, attention).to(torch.bfloat16)
    w_o, w_gate_up, w_down = ((normal(rows, cols) / cols ** 0.5).to(torch.bfloat16)
                              for rows, cols in ((hidden, attention), (2 * inter, hidden), (hidden, inter)))
    base, weight = normal(m, hidden), 1 + 0.3 * normal(hidden)
    o, gate_up, down = K.pack_weight(w_o), K.pack_weight(w_gate_up), K.pack_weight(w_down)
    residual64 = base.double() + attended.double() @ w_o.double().t()
    normed64 = residual64 / torch.sqrt((residual64 ** 2).mean(-1, keepdim=True) + 1e-5) * weight.double()
    both = normed64 @ w_gate_up.double().t()
    want = residual64 + (both[:, :inter] / (1 + torch.exp(-both[:, :inter])) * both[:, inter:]) @ w_down.double().t()
    for reader in (None, ProductReader(inter, True)):
        residual = base.clone()
        x = K.gemm(attended, o, residual, accumulate=True, then_norm=NormRequest(weight, 1e-5, reader))
        if x is None:
            x = K.new_rows(m, hidden, torch.bfloat16, inter, True)
            K.rmsnorm(residual, weight, 1e-5, x)
        activated = K.new_rows(m, inter, torch.bfloat16, hidden)
        K.gemm_swiglu(x, gate_up, activated)
        K.gemm(activated, down, residual, accumulate=True)
        # three bfloat16 roundings on the way (the norm's rows, the gated output, and once more where a norm rides)
        assert rel(residual, want.cpu()) < 1e-2
