"""Recurrences with a scalar decay as products of matrices over chunks of 64 rows, against the recurrence in float64: sequences that
end at, before and after a chunk's end, sequences of one row beside long ones, more chunks than their states have memory for at once."""

import numpy as np
import pytest
import torch

from test_gpu_kernels import K, dev      # noqa: F401  (K: the fixture)

pytestmark = pytest.mark.gpu


def recurrence(state, q, k, v, decay, weight, skip):
    """state [H, D, V], q, k [T, H, D], v [T, H, V], decay, weight [T, H], skip [H], all float64 on the device."""
    out = torch.empty_like(v)
    for t in range(len(q)):
        state = decay[t][:, None, None] * state + weight[t][:, None, None] * k[t][:, :, None] * v[t][:, None, :]
        out[t] = (q[t][:, None, :] @ state)[:, 0] + skip[:, None] * v[t]
    return out, state


def close(got, want):
    # 32-bit sums of D products and of the chunk's rows, then one product and sum a chunk: far below 256 roundings of the largest
    return float((got.double() - want).abs().max()) <= 256 * 2.0 ** -24 * float(want.abs().max())


LENGTHS = [[128], [129, 1, 127, 64], [130, 64, 1, 1, 192], [1] * 70 + [128, 65, 300]]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads,dim,vdim,decay,lengths", [
    (1, 64, 16, [0.97], LENGTHS[0]), (3, 96, 48, [0.999, 0.4, 1.0], LENGTHS[1]), (2, 128, 128, [0.0, 0.9], LENGTHS[2]),
    (2, 64, 64, [-0.7, 1.001], LENGTHS[3]), (64, 128, 128, list(np.linspace(0.5, 0.9999, 64)), [1700, 3, 900])])
def test_lightning_scan_as_products(K, dtype, heads, dim, vdim, decay, lengths):
    keys, values = heads * dim, heads * vdim
    stride = 2 * keys + 2 * values
    assert K.lib.bh_lightning_products_scratch(len(lengths), sum(lengths), max(lengths), heads, dim, vdim, stride, 0, keys, 2 * keys) > 0
    g = torch.Generator().manual_seed(heads + dim + len(lengths))
    slots = torch.randperm(len(lengths) + 2, generator=g)[:len(lengths)]
    state = torch.randn(len(lengths) + 2, heads, dim, vdim, generator=g).cuda()      # an earlier step's, and slots of nobody here
    before = state.clone()
    proj = torch.randn(sum(lengths), stride, generator=g).to(dtype).cuda()
    starts = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    factors = torch.tensor(decay, dtype=torch.float32)
    out = torch.full((sum(lengths), values), float("nan"), device="cuda:0")
    K.lightning_scan(proj, 0, keys, 2 * keys, state, dev(factors), dev(torch.from_numpy(starts)), dev(slots.to(torch.int32)), out,
                     heads, dim, vdim, max_rows_per_seq=max(lengths))
    opened = torch.nn.functional.silu(proj.double())
    for b, slot in enumerate(slots.tolist()):
        rows = opened[starts[b]:starts[b + 1]]
        q, k, v = (rows[:, lo:lo + heads * n].reshape(-1, heads, n) for lo, n in ((0, dim), (keys, dim), (2 * keys, vdim)))
        ones = torch.ones(len(rows), heads, dtype=torch.float64, device="cuda:0")
        want, last = recurrence(before[slot].double(), q, k, v, ones * factors.double().cuda(), ones, torch.zeros(heads, dtype=torch.float64, device="cuda:0"))
        assert close(out[starts[b]:starts[b + 1]], want.reshape(len(rows), -1)), (b, len(rows))
        assert close(state[slot], last), (b, len(rows))
    untouched = [s for s in range(len(lengths) + 2) if s not in slots.tolist()]
    assert torch.equal(state[untouched], before[untouched])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads,groups,vdim,n_state,rates,lengths", [
    (2, 1, 16, 64, (-2.5, 0.5), LENGTHS[0]), (6, 3, 48, 96, (-2.5, 0.5), LENGTHS[1]), (4, 4, 64, 128, (3.0, 12.0), LENGTHS[2]),
    (8, 2, 64, 64, (-9.0, -8.0), LENGTHS[3]), (160, 8, 64, 128, (-1.0, 2.0), [1500, 2, 700])])
def test_state_space_scan_as_products(K, dtype, heads, groups, vdim, n_state, rates, lengths):
    """Decays from almost none to rows that forget everything."""
    inner, total = heads * vdim, sum(lengths)
    g = torch.Generator().manual_seed(heads + n_state + len(lengths))
    xbc = torch.randn(total, inner + 2 * groups * n_state, generator=g).cuda()
    proj = torch.randn(total, heads + 4, generator=g).to(dtype).cuda()
    bias = (torch.rand(heads, generator=g) * 4 - 3).cuda()
    a_log = (torch.rand(heads, generator=g) * (rates[1] - rates[0]) + rates[0]).cuda()
    skip = torch.randn(heads, generator=g).cuda()
    size, tail = heads * n_state * vdim, 12
    assert K.lib.bh_ssm_products_scratch(len(lengths), total, max(lengths), heads, vdim, n_state, groups, xbc.shape[1]) > 0
    state = torch.randn(len(lengths) + 1, size + tail, generator=g).cuda()
    before = state.clone()
    slots = torch.randperm(len(lengths) + 1, generator=g)[:len(lengths)]
    starts = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    out = torch.full((total, inner), float("nan"), device="cuda:0")
    K.ssm_scan(xbc, proj, 4, bias, a_log, skip, state, 0, dev(torch.from_numpy(starts)), dev(slots.to(torch.int32)), out, heads, vdim,
               n_state, groups, max_rows_per_seq=max(lengths))
    dt = torch.nn.functional.softplus(proj[:, 4:].double() + bias.double(), threshold=30)
    decay = torch.exp(-torch.exp(a_log.double()) * dt)
    x = xbc[:, :inner].double().reshape(total, heads, vdim)
    b, c = (xbc[:, lo:lo + groups * n_state].double().reshape(total, groups, n_state).repeat_interleave(heads // groups, 1)
            for lo in (inner, inner + groups * n_state))
    for i, slot in enumerate(slots.tolist()):
        rows = slice(starts[i], starts[i + 1])
        want, last = recurrence(before[slot, :size].double().reshape(heads, n_state, vdim), c[rows], b[rows], x[rows], decay[rows], dt[rows], skip.double())
        assert close(out[rows], want.reshape(-1, inner)), (i, lengths[i])
        assert close(state[slot, :size].reshape(heads, n_state, vdim), last), (i, lengths[i])
    assert torch.equal(state[:, size:], before[:, size:])


def test_scans_of_sizes_that_are_no_whole_tiles_keep_their_walk(K):
    for heads, dim, vdim in ((2, 48, 64), (2, 32, 64), (2, 64, 24), (1, 64, 272), (1, 320, 256)):
        assert K.lib.bh_lightning_products_scratch(1, 500, 500, heads, dim, vdim, 4096, 0, 1024, 2048) == 0
    assert K.lib.bh_lightning_products_scratch(1, 500, 500, 2, 64, 64, 514, 0, 128, 256) == 0       # rows that lie on no 16 bytes
    assert K.lib.bh_lightning_products_scratch(8, 8, 1, 2, 64, 64, 512, 0, 128, 256) == 0           # a decode step


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
@pytest.mark.parametrize("row", [0, 16, 37, 63, 64, 111, 190, 199])
@pytest.mark.parametrize("kind", ["lightning", "state space"])
def test_a_value_that_is_not_finite_reaches_no_earlier_row(K, kind, row, value):
    """The rows before it, the other columns' rows, heads and sequences have the bits that they have without it; its own row and the
    later ones are not finite in its column, as in the recurrence."""
    heads, dim, vdim, lengths, column = 2, 64, 48, [200, 130], 21
    total, width = sum(lengths), heads * vdim
    g = torch.Generator().manual_seed(row)
    starts, slots = dev(torch.tensor([0, 200, 330], dtype=torch.int32)), dev(torch.tensor([1, 0], dtype=torch.int32))
    keys = heads * dim
    rows = torch.randn(total, 2 * keys + width, generator=g).cuda()      # q, k, v, or v, k, q
    rates, state = torch.randn(total, heads, generator=g).cuda(), torch.randn(2, heads, dim, vdim, generator=g).cuda()
    first = 2 * keys if kind == "lightning" else 0

    def run(rows):
        out, held = torch.full((total, width), 7.0, device="cuda:0"), state.clone()
        if kind == "lightning":
            K.lightning_scan(rows, 0, keys, 2 * keys, held, dev(torch.tensor([0.9, 0.99])), starts, slots, out, heads, dim, vdim, max_rows_per_seq=200)
        else:
            zero = torch.zeros(heads, device="cuda:0")
            K.ssm_scan(rows, rates, 0, zero - 2.0, zero, zero + 1.0, held.view(2, -1), 0, starts, slots, out, heads, vdim, dim, heads, max_rows_per_seq=200)
        return out, held

    assert K.lib.bh_lightning_products_scratch(2, total, 200, heads, dim, vdim, rows.shape[1], 0, keys, 2 * keys) > 0
    assert K.lib.bh_ssm_products_scratch(2, total, 200, heads, vdim, dim, heads, rows.shape[1]) > 0
    clean, _ = run(rows)
    spoilt = rows.clone()
    spoilt[row, first + vdim + column] = value      # head 1
    got, held = run(spoilt)
    at = vdim + column
    assert torch.isfinite(clean).all() and not torch.isfinite(got[row:200, at]).any()
    assert not torch.isfinite(held[1, 1, :, column]).any()
    got[row:200, at] = clean[row:200, at]
    assert torch.equal(got, clean)


@pytest.mark.parametrize("first", [63, 64, 70, 200])
def test_scans_of_sequences_that_start_behind_the_step_s_first_row(K, first):
    """Rows before the first sequence belong to nobody: neither read nor written."""
    heads, dim, vdim, lengths = 2, 64, 64, [150, 1, 128]
    total, keys, width = first + sum(lengths), heads * dim, heads * vdim
    g = torch.Generator().manual_seed(first)
    rows = torch.randn(total, 2 * keys + width, generator=g).cuda()
    rows[:first] = float("nan")
    rates, state = torch.randn(total, heads, generator=g).cuda(), torch.randn(3, heads, dim, vdim, generator=g).cuda()
    starts = np.concatenate([[first], first + np.cumsum(lengths)]).astype(np.int32)
    slots, zero = dev(torch.tensor([2, 0, 1], dtype=torch.int32)), torch.zeros(heads, device="cuda:0")
    for shift in (0, first):      # as they lie, and without those rows
        at = dev(torch.from_numpy(starts - shift))
        outs = [torch.full((total - shift, width), 7.0, device="cuda:0") for _ in range(2)]
        held = [state.clone() for _ in range(2)]
        K.lightning_scan(rows[shift:].contiguous(), 0, keys, 2 * keys, held[0], dev(torch.tensor([0.9, 0.99])), at, slots, outs[0], heads, dim, vdim,
                         max_rows_per_seq=150)
        K.ssm_scan(rows[shift:].contiguous(), rates[shift:].contiguous(), 0, zero - 2.0, zero, zero + 1.0, held[1].view(3, -1), 0, at, slots, outs[1],
                   heads, vdim, dim, heads, max_rows_per_seq=150)
        if shift == 0:
            behind = outs, held
    for a, b in zip(behind[0], outs):
        assert bool((a[:first] == 7.0).all()) and torch.isfinite(b).all() and torch.equal(a[first:], b)
    for a, b in zip(behind[1], held):
        assert torch.equal(a, b)
