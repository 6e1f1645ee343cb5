"""The experts' products of many pairs (`experts_many`) against float64, where tiles of pairs, blocks of weight rows and the search
for a workgroup's tile end."""

import pytest
import torch

from test_gpu_kernels import K, dev      # noqa: F401  (K: the fixture)

pytestmark = pytest.mark.gpu


# pairs an expert: none, one, a tile's edges (64 and 128), several tiles; experts: one, more than a wave's lanes; outputs: less than
# a tile's, remainders of one; widths of 1 to 5, 7, 12 and 32 units of 64 k, the ring of three units among them; so few workgroups run on
# tiles of 64 pairs
@pytest.mark.parametrize("counts,width,ff", [([1], 64, 64), ([64, 0, 65, 1], 128, 192), ([0, 63, 127, 0, 30], 192, 64), ([300], 64, 128),
                                             ([128, 129, 127, 257, 0], 256, 64), ([0] * 69 + [200, 3] + [0] * 5 + [40], 64, 64),
                                             ([150] * 66, 64, 64), ([97, 512], 2048, 768),
                                             ([130, 5], 320, 448), ([33, 70, 2], 448, 320)])
@pytest.mark.parametrize("weighed", [False, True])
def test_experts_of_many_pairs(K, counts, width, ff, weighed):
    g = torch.Generator().manual_seed(sum(counts) + width)
    experts, pairs = len(counts), sum(counts)
    x = torch.randn(pairs, width, generator=g).bfloat16()             # one pair a row
    gate_up = (torch.randn(experts, 2 * ff, width, generator=g) / width ** 0.5).bfloat16()
    down = (torch.randn(experts, width, ff, generator=g) / ff ** 0.5).bfloat16()
    order = torch.randperm(pairs, generator=g)
    lists, at, owner = torch.zeros(experts, pairs, dtype=torch.int32), 0, torch.empty(pairs, dtype=torch.long)
    for e, count in enumerate(counts):
        lists[e, :count] = order[at:at + count].to(torch.int32)
        owner[order[at:at + count]] = e
        at += count
    shares = torch.rand(pairs, 1, generator=g) + 0.5
    held = dev(torch.tensor(counts, dtype=torch.int32))
    inner = torch.full((pairs, ff), float("nan"), dtype=torch.bfloat16, device="cuda:0")
    K.experts_many(dev(x), 1, dev(lists), held, K.pack_weight(dev(gate_up.reshape(-1, width))), inner, gated=True, limit=1.5, alpha=1.702,
                   shift=1.0, **({"in_weights": dev(shares)} if weighed else {}))
    out = torch.full((pairs, width), float("nan"), device="cuda:0")
    K.experts_many(inner, 1, dev(lists), held, K.pack_weight(dev(down.reshape(-1, ff))), out)
    got_inner, got = inner.cpu().double(), out.cpu().double()
    for e in range(experts):
        rows = (owner == e).nonzero()[:, 0]
        if not len(rows):
            continue
        both = x[rows].double() @ gate_up[e].double().T * (shares[rows].double() if weighed else 1.0)
        gate, up = both[:, :ff].clamp(max=1.5), both[:, ff:].clamp(-1.5, 1.5)
        want = gate * torch.sigmoid(1.702 * gate) * (up + 1.0)
        # the result is rounded to 8 bits; the sums' own error (float32) is far below that
        assert float(((got_inner[rows] - want).abs() - 2.0 ** -8 * want.abs()).max()) < 1e-4, e
        want = got_inner[rows] @ down[e].double().T
        assert float((got[rows] - want).abs().max()) < 2.0 ** -24 * (ff + 8) * float((got_inner[rows].abs() @ down[e].double().abs().T).max()), e


# more workgroups than a round holds, on tiles of 128 pairs: one beyond and one short of a tile, empty and lone ones; 1, 2, 3, 5 and 7 units
# of 64 k on either product
@pytest.mark.parametrize("repeats,width,ff,both", [(9, 64, 512, False), (9, 128, 576, False), (9, 192, 512, False), (9, 320, 448, True),
                                                   (18, 448, 320, True), (20, 320, 64, True), (20, 320, 128, True), (20, 384, 192, True)])
def test_experts_of_many_pairs_in_tiles_of_128(K, repeats, width, ff, both):
    counts = [130, 5, 64, 128, 129, 257, 0, 127] * repeats
    assert K.lib.bh_experts_many_tile(sum(counts), len(counts), width, ff, 1) == 128
    assert not both or K.lib.bh_experts_many_tile(sum(counts), len(counts), ff, width, 0) == 128
    test_experts_of_many_pairs(K, counts, width, ff, False)


def test_experts_of_many_pairs_take_rows_shared_by_choices(K):
    """A row's pairs read the same input: pair p reads row p // top."""
    g = torch.Generator().manual_seed(3)
    top, rows, width, ff = 3, 70, 64, 64
    x = torch.randn(rows, width, generator=g).bfloat16()
    w = (torch.randn(2 * ff, width, generator=g) / 8).bfloat16()
    lists = torch.arange(rows * top, dtype=torch.int32)[None]
    inner = torch.empty(rows * top, ff, dtype=torch.bfloat16, device="cuda:0")
    K.experts_many(dev(x), top, dev(lists), dev(torch.tensor([rows * top], dtype=torch.int32)), K.pack_weight(dev(w)), inner, gated=True,
                   limit=float("inf"), alpha=1.0, shift=0.0)
    both = x.double() @ w.double().T
    want = (torch.nn.functional.silu(both[:, :ff]) * both[:, ff:]).repeat_interleave(top, 0)
    assert float(((inner.cpu().double() - want).abs() - 2.0 ** -8 * want.abs()).max()) < 1e-4
