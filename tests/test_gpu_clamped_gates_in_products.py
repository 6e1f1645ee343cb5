"""A clamped gate in its product, and a norm's output in rows and in blocks, against float64."""

import pytest
import torch

from test_gpu_kernels import K, dev, rel      # noqa: F401  (K: the fixture)

pytestmark = pytest.mark.gpu


# What goes in one piece of many rows, of the sizes below.
MANY_ROWS = [(2100, 768, 1024), (300, 3072, 2048), (2100, 3072, 2048), (300, 4096, 256), (2100, 4096, 256)]


# rows: every kernel that gates (up to 8, 16 and 32 rows, 33 to 96, whole tiles, many rows); outputs: one block, blocks that fill no round, many
@pytest.mark.parametrize("m", [1, 8, 9, 16, 31, 33, 64, 100, 128, 129, 300, 2100])
@pytest.mark.parametrize("ff,k", [(16, 64), (48, 512), (768, 1024), (3072, 2048), (4096, 256)])
@pytest.mark.parametrize("blocks", [False, True])
def test_clamped_gate_in_a_product(K, m, ff, k, blocks):
    g = torch.Generator().manual_seed(m + ff + k)
    a, w = (torch.randn(rows, k, generator=g).to(torch.bfloat16) for rows in (m, 2 * ff))
    w = (w.float() * (3.0 / k ** 0.5)).to(torch.bfloat16)      # gates and ups of about 3: a fifth of them beyond the limit
    out = K.new_rows(m, ff, torch.bfloat16, 1024) if blocks else torch.full((m, ff), float("nan"), dtype=torch.bfloat16, device="cuda:0")
    took = K.gemm_clamped_glu(dev(a), K.pack_weight(dev(w)), out, 4.0, 1.702)
    assert took is (m <= 32 or (m, ff, k) in MANY_ROWS)
    if not took:      # (the two launches do it then)
        return
    compare(K, a, w, out)


def compare(K, a, w, out):
    ff, k = w.shape[0] // 2, w.shape[1]
    both = a.double() @ w.double().T
    gate, up = both[:, :ff].clamp(max=4.0), both[:, ff:].clamp(-4.0, 4.0)
    want = gate * torch.sigmoid(1.702 * gate) * (up + 1.0)
    got = out if isinstance(out, torch.Tensor) else K.from_blocked(out)
    # half a unit of the result's 8 bits, and float32 sums of k products whose error the gate and up pass on at most 5-fold
    bound = 2.0 ** -8 * want.abs() + 8 * (k / 16 + 64) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T)[:, :ff] + 1e-5
    assert bool(((got.cpu().double() - want).abs() <= bound).all())


# the smallest sizes that each tile of many rows takes: 128 x 128, the same with k in halves, 256 x 128, and those whose waves load in turns, 256 x 192 and 256 x 256
@pytest.mark.parametrize("tile,m,ff,k", [(0, 257, 512, 128), (1, 700, 1024, 4096), (2, 257, 6144, 128), (3, 700, 6144, 128), (4, 1100, 5120, 128)])
def test_clamped_gate_in_each_tile_of_many_rows(K, tile, m, ff, k):
    assert K.lib.bh_gemm_bf16_plan(m, ff, k, 1, 1) == 16 * tile + 1
    g = torch.Generator().manual_seed(tile)
    a, w = torch.randn(m, k, generator=g).to(torch.bfloat16), (torch.randn(2 * ff, k, generator=g) * (3.0 / k ** 0.5)).to(torch.bfloat16)
    for out in (torch.full((m, ff), float("nan"), dtype=torch.bfloat16, device="cuda:0"), K.new_rows(m, ff, torch.bfloat16, 1024)):
        assert K.gemm_clamped_glu(dev(a), K.pack_weight(dev(w)), out, 4.0, 1.702)
        compare(K, a, w, out)


def test_not_a_numbers_go_as_in_the_activation_of_its_own(K):
    a, w = torch.randn(4, 64).to(torch.bfloat16), torch.randn(64, 64).to(torch.bfloat16)
    a[1, 3], a[2, 5], a[3, 0] = float("nan"), float("inf"), float("-inf")
    packed, out, both, apart = K.pack_weight(dev(w)), torch.empty(4, 32, dtype=torch.bfloat16, device="cuda:0"), torch.empty(4, 64, dtype=torch.bfloat16, device="cuda:0"), None
    assert K.gemm_clamped_glu(dev(a), packed, out, 7.0, 1.702)
    K.gemm(dev(a), packed, both)
    apart = torch.empty_like(out)
    K.clamped_glu(both, apart, 7.0, 1.702)
    assert torch.equal(out.isfinite(), apart.isfinite()) and rel(out.nan_to_num(0, 0, 0), apart.nan_to_num(0, 0, 0).double()) < 2e-2
    assert K.gemm_clamped_glu(dev(a), packed, out, 0.0, 1.702) is False and K.gemm_clamped_glu(dev(a), dev(w), out, 7.0, 1.702) is False


@pytest.mark.parametrize("rows,width", [(1, 64), (5, 96), (8, 2048), (16, 1024), (33, 512), (300, 2048), (7, 34), (40, 20480)])
def test_norms_in_rows_and_blocks(K, rows, width):
    from beholdd.kernels.library import BothRows
    x, weight, bias = torch.randn(rows, width), torch.randn(width), torch.randn(width)
    out = K.new_both_rows(rows, width, torch.bfloat16, 1024)
    if not isinstance(out, BothRows):
        assert width % 64 or rows > 32      # (a product of these sizes reads rows)
        return
    out.row_by_row.fill_(float("nan"))
    K.layernorm(dev(x), dev(weight), dev(bias), 1e-5, out)
    alone = torch.empty(rows, width, dtype=torch.bfloat16, device="cuda:0")
    K.layernorm(dev(x), dev(weight), dev(bias), 1e-5, alone)
    assert torch.equal(out.row_by_row, alone) and torch.equal(K.from_blocked(out.blocks), alone)
    for matrix in (torch.randn(96, width), torch.randn(33, width)):      # and products read it, packed and not
        w = dev(matrix.to(torch.bfloat16))
        for form in (K.pack_weight(w), w):
            got, want = torch.empty(rows, len(matrix), device="cuda:0"), torch.empty(rows, len(matrix), device="cuda:0")
            K.gemm(out, form, got)
            K.gemm(alone, form, want)
            assert rel(got, want.double()) < 1e-5
