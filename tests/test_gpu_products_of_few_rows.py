"""Products of up to 32 rows of packed weights at the edges of what a workgroup owns and a wave holds, against float64."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    from beholdd.kernels import HipKernels
    return HipKernels()


def rel(got, want):
    return float((got.double() - want).abs().max() / want.abs().max())


# k: waves without a chunk, one and two chunks a wave and one more or less (all at once / in turn), the same for the four sets of the
# spans of 8 rows (n of up to 2,048 from k of 1,536 on); n: spans of 16, 8, 20 and 24 rows, an odd number of workgroups, more than four
# workgroups a compute unit and long k at more than 16 rows (the kernel that asks in bursts)
@pytest.mark.parametrize("n,k", [(96, 64), (4096, 512), (2064, 960), (4080, 1024), (4112, 1088), (16, 1536), (1040, 1984), (2048, 2048),
                                 (2032, 2112), (336, 5184), (5120, 448), (5120, 2112), (6144, 1024), (6144, 4160), (17408, 256), (2560, 2112)])
@pytest.mark.parametrize("m", [1, 8, 9, 16, 17, 32])
def test_products_of_few_rows(K, m, n, k):
    """float32 with and without accumulation and a norm behind, bfloat16 behind prepared norm rows, squared, and gated, from rows and
    from blocks whose rows behind the last hold NaN; the bounds are those of a sum of k float32 products and of bfloat16 roundings."""
    from beholdd.kernels.library import BlockedRows
    from beholdd.parts.base import NormRequest
    g = torch.Generator(device="cuda:0").manual_seed(m + n + k)
    normal = lambda *shape: torch.randn(*shape, generator=g, device="cuda:0")
    a, w = normal(m, k).to(torch.bfloat16), (normal(n, k) / k ** 0.5).to(torch.bfloat16)
    packed, block_rows = K.pack_weight(w), int(K.lib.bh_gemm_bf16_reads_blocked(m, n, k, 1, 0))
    assert block_rows == (8 if m <= 8 else 16)
    x = BlockedRows(torch.full((BlockedRows.padded_rows(m, block_rows) * k,), float("nan"), dtype=torch.bfloat16, device="cuda:0"), m, k, block_rows)
    K.to_blocked(a, x, block_rows)
    want, bound = a.double() @ w.double().t(), 4 * math.sqrt(k) * 2.0 ** -24
    empty = lambda dtype: torch.full((m, n), float("nan"), dtype=dtype, device="cuda:0")
    out = empty(torch.float32)
    K.gemm(x, packed, out)
    assert rel(out, want) < bound
    stream = torch.cuda.current_stream().cuda_stream
    direct = empty(torch.float32)      # rows one after the other, which the entry takes as well
    assert K.lib.bh_gemm_bf16(a.data_ptr(), packed.data.data_ptr(), direct.data_ptr(), 0, 0, m, n, k, 1, 0, None, 0, 0.0, None, 0, None, None, None,
                              0, 0, 0, stream) == 0
    assert torch.equal(direct, out)
    base, weight, eps = normal(m, n), 1 + 0.3 * normal(n), 1e-5
    total = base.clone()
    prepared = K.gemm(x, packed, total, accumulate=True, then_norm=NormRequest(weight, eps))
    assert rel(total, want + base.double()) < bound
    assert rel(prepared.ss.sum(1), (total.double() ** 2).sum(-1)) < 1e-5
    assert rel(prepared.rows, total.double() * weight.double()) < 4e-3
    # prepared rows of width n in front of products of this shape turned round: the row factor
    w2 = (normal(160, n) / n ** 0.5).to(torch.bfloat16)
    if n % 64 == 0:
        normed = total.double() / torch.sqrt((total.double() ** 2).mean(-1, keepdim=True) + eps) * weight.double()
        rounded = torch.empty(m, 160, dtype=torch.bfloat16, device="cuda:0")
        K.gemm(prepared, K.pack_weight(w2), rounded)
        assert rel(rounded, normed @ w2.double().t()) < 1e-2
    for rows in (0, block_rows) if n % 32 == 0 else (0,):
        squared = empty(torch.bfloat16) if not rows else K.to_blocked(empty(torch.bfloat16), block_rows=rows)
        if K.gemm_relu_squared(x, packed, squared):
            assert rel(K.from_blocked(squared) if rows else squared, want.clamp(min=0) ** 2) < 4e-3 + 4 * bound
    up = (normal(n, k) / k ** 0.5).to(torch.bfloat16)
    gated = empty(torch.bfloat16)
    K.gemm_swiglu(x, K.pack_weight(torch.cat([w, up])), gated)
    assert rel(gated, want / (1 + torch.exp(-want)) * (a.double() @ up.double().t())) < 6e-3


# rows around the groups of four and the last of the few; k: shorter than a wave's load, remainders of a chunk and of a trip, eight waves;
# outputs: every split of a workgroup's rows
@pytest.mark.parametrize("m,n,k", [(1, 5, 60), (3, 64, 64), (4, 2048, 1024), (5, 7, 68), (8, 4099, 256), (9, 130, 516), (16, 8200, 132),
                                   (17, 33, 2052), (31, 516, 3072), (32, 16, 2048), (32, 1030, 1088)])
def test_float32_products_norm_a_residual(K, m, n, k):
    """A float32 product leaves the norm behind it to the product that reads it; both together against float64.  The bound: a sum of k
    products, each of which is off by the roundings of its factors (the weight's, the row factor's with its sum of squares)."""
    from beholdd.kernels import NormedRows
    from beholdd.parts.base import NormRequest
    g = torch.Generator(device="cuda:0").manual_seed(m + n + k)
    normal = lambda *shape: torch.randn(*shape, generator=g, device="cuda:0")
    a, w_in, w, weight, eps = normal(m, 64), normal(k, 64) / 8, normal(2 * n, k) / k ** 0.5, 1 + 0.3 * normal(k), 1e-5
    residual = normal(m, k)
    want_residual = residual.double() + a.double() @ w_in.double().t()
    prepared = K.gemm(a, w_in, residual, accumulate=True, then_norm=NormRequest(weight, eps))
    assert isinstance(prepared, NormedRows) and prepared.ss is None and rel(residual, want_residual) < 64 * 2.0 ** -24
    source = residual.double()
    normed = source / torch.sqrt((source ** 2).mean(-1, keepdim=True) + eps) * weight.double()
    bound = (k / 16 + 72) * 2.0 ** -24 * (normed.abs() @ w.double().abs().t())
    out = torch.full((m, n), float("nan"), device="cuda:0")
    half = w[:n].contiguous()
    assert K.gemm(prepared, half, out) is None
    assert bool(((out.double() - normed @ half.double().t()).abs() <= bound[:, :n]).all())
    gated = torch.full((m, n), float("nan"), device="cuda:0")
    K.gemm_swiglu(prepared, w, gated)
    both = normed @ w.double().t()
    gate, up = both[:, :n], both[:, n:]
    # d(silu) is at most 1.1, and the function itself some roundings
    slack = 1.1 * bound[:, :n] * up.abs() + bound[:, n:] * gate.abs() + 16 * 2.0 ** -24 * (gate * up).abs() + 1e-30
    assert bool(((gated.double() - gate / (1 + torch.exp(-gate)) * up).abs() <= slack).all())
    # one that adds to what is there runs the norm as a launch of its own
    total = normal(m, n)
    base = total.double()
    K.gemm(prepared, half, total, accumulate=True)
    assert bool(((total.double() - base - normed @ half.double().t()).abs() <= bound[:, :n] + 4 * 2.0 ** -24 * base.abs()).all())


def test_float32_products_norm_without_an_epsilon(K):
    """A norm's epsilon may be zero, as `rmsnorm` takes it, and one below the smallest float32 is."""
    from beholdd.parts.base import NormRequest
    g = torch.Generator(device="cuda:0").manual_seed(5)
    a, w_in, w, weight = (torch.randn(*shape, generator=g, device="cuda:0") for shape in ((4, 64), (256, 64), (24, 256), (256,)))
    for eps in (0.0, 1e-60):
        residual = torch.randn(4, 256, generator=g, device="cuda:0")
        prepared = K.gemm(a, w_in, residual, accumulate=True, then_norm=NormRequest(weight, eps))
        assert prepared.ss is None
        source = residual.double()
        normed = source / source.square().mean(-1, keepdim=True).sqrt() * weight.double()
        out, gated = torch.empty(4, 24, device="cuda:0"), torch.empty(4, 12, device="cuda:0")
        K.gemm(prepared, w, out)
        K.gemm_swiglu(prepared, w, gated)
        both = normed @ w.double().t()
        bound = (256 / 16 + 72) * 2.0 ** -24 * float((normed.abs() @ w.double().abs().t()).max())
        assert float((out.double() - both).abs().max()) < bound
        assert float((gated.double() - torch.nn.functional.silu(both[:, :12]) * both[:, 12:]).abs().max()) < 3 * bound * float(both.abs().max())


@pytest.mark.parametrize("n,first", [(512, 0), (256, 2048), (256, 0)])
def test_float32_products_may_overwrite_what_they_norm(K, n, first):
    """The output on the residual itself, on its last elements and on its first: the norm is then a launch of its own."""
    from beholdd.parts.base import NormRequest
    g = torch.Generator(device="cuda:0").manual_seed(n + first)
    m, k = 8, 512
    a, w_in, w, weight = (torch.randn(*shape, generator=g, device="cuda:0") for shape in ((m, 64), (k, 64), (n, k), (k,)))
    residual = torch.randn(m, k, generator=g, device="cuda:0")
    prepared = K.gemm(a, w_in, residual, accumulate=True, then_norm=NormRequest(weight, 1e-5))
    source = residual.double()
    want = source / (source.square().mean(-1, keepdim=True) + 1e-5).sqrt() * weight.double() @ w.double().t()
    out = residual.view(-1)[first:first + m * n].view(m, n)
    K.gemm(prepared, w, out)
    assert float((out.double() - want).abs().max()) < (k / 16 + 72) * 2.0 ** -24 * float(want.abs().max()) * 8


# rows and outputs on both sides of each line of the rule (bh_gemm_f32_takes_norm): gated products stop at half as many outputs as plain ones
@pytest.mark.parametrize("m,n,k,plain,gated", [(4, 8200, 132, 1, 1), (1, 8192, 68, 1, 1), (8, 4095, 260, 1, 1), (5, 4096, 64, 1, 0), (16, 8191, 64, 1, 0),
                                               (9, 8192, 64, 0, 0), (17, 1024, 768, 1, 1), (32, 1025, 64, 0, 0), (24, 8, 772, 0, 0)])
def test_float32_products_that_norm_and_those_that_leave_it(K, m, n, k, plain, gated):
    takes = K.lib.bh_gemm_f32_takes_norm
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:      # the lines go by the compute units
        assert (takes(m, n, k, 0), takes(m, n, k, 1)) == (plain, gated)
    test_float32_products_norm_a_residual(K, m, n, k)
