"""Walks of many rows whose threads keep two columns of the state, at the sizes where their tiles, stages and chunks end, against plain sums
in 64 bits.  A walk adds up to 256 products of 32-bit numbers a row and carries the state on, which the tests of the other walks bound by
2e-5 as well."""

import numpy as np
import pytest
import torch

import plain_vitudra as plain
from test_gpu_pudorax import dev, ragged, rel, rounded

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16]


@pytest.fixture(scope="module")
def K():
    from beholdd.kernels import HipKernels
    return HipKernels("cuda:0")


def gla_recurrence(q, k, v, a, state):
    s = np.zeros((q.shape[1], q.shape[2], v.shape[2])) if state is None else state.copy()
    o = np.zeros_like(v)
    for t in range(len(q)):
        s = a[t][:, :, None] * s + k[t][:, :, None] * v[t][:, None, :]
        o[t] = np.einsum("hdv,hd->hv", s, q[t])
    return o, s


APART = [(260, 34, 34), (3, 64, 64), (300, 64, 64), (130, 132, 44)]      # what stays with the other walk of the sizes below


# the sizes of a column's lanes (up to 64, 128, 256 key dimensions), tiles that values do not fill, stages and chunks that end early, sequences of
# one row beside long ones; columns that are no multiple of four, few workgroups and short sequences stay with the other walk
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rule", ["wkv", "gla"])
@pytest.mark.parametrize("heads,dim,vdim,lengths", [(64, 64, 64, [300, 17, 1, 64]), (260, 36, 36, [65]), (70, 68, 100, [79, 3, 90]), (130, 132, 44, [70]), (64, 256, 260, [66]),
                                                    (260, 132, 44, [70]), (16, 128, 128, [1000, 5]), (9, 256, 252, [1000]), (33, 100, 64, [300, 260]),      # the last three in chunks
                                                    (260, 34, 34, [65]), (3, 64, 64, [200]), (300, 64, 64, [63, 5])])
def test_walks_in_columns(K, dtype, rule, heads, dim, vdim, lengths):
    if rule == "wkv":
        vdim = dim
    assert bool(K.lib.bh_gla_in_columns(len(lengths), max(lengths), heads, dim, vdim)) is ((heads, dim, vdim) not in APART)
    rng = np.random.default_rng(heads * dim + vdim)
    n, kw, vw, slots = sum(lengths), heads * dim, heads * vdim, len(lengths) + 1
    order = [int(i) for i in rng.permutation(slots)[:len(lengths)]]
    seq_start, seq_slot, _, starts = ragged(lengths, order)
    bias, bonus = rng.uniform(-6, 0, kw).astype(np.float32), rng.standard_normal(kw).astype(np.float32)
    state, held = torch.zeros(slots, kw * vdim, device="cuda:0"), [None] * len(lengths)
    for step in range(2):
        rows_t, rows = rounded(rng.standard_normal((n, 2 * kw + vw)), dtype)
        z = rng.standard_normal((n, kw)).astype(np.float32)
        out = torch.full((n, vw), 9.0, device="cuda:0")
        if rule == "wkv":
            K.wkv_scan(*(dev(rows_t[:, i * kw:(i + 1) * kw].contiguous()) for i in range(3)), dev(z), dev(bias), dev(bonus), state, 0, seq_start, seq_slot, out,
                       heads, dim, vdim, max_rows_per_seq=max(lengths))
        else:
            K.gla_scan(dev(rows_t), 0, kw, 2 * kw, dev(z), dev(bias), 8.0, dim ** -0.5, state.view(slots, heads, dim, vdim), seq_start, seq_slot, out, heads, dim, vdim,
                       max_rows_per_seq=max(lengths))
        for s, length in enumerate(lengths):
            lo = starts[s]
            here = rows[lo:lo + length].astype(np.float64)
            q, k = (here[:, i * kw:(i + 1) * kw].reshape(length, heads, dim) for i in range(2))
            v, x = here[:, 2 * kw:].reshape(length, heads, vdim), (z[lo:lo + length].astype(np.float64) + bias).reshape(length, heads, dim)
            if rule == "wkv":
                want, held[s] = plain.wkv_recurrence(q, k, v, np.exp(-np.exp(x)), bonus.reshape(heads, dim), state=held[s])
            else:
                want, held[s] = gla_recurrence(q * dim ** -0.5, k, v, (1 / (1 + np.exp(-x))) ** (1 / 8.0), held[s])
            assert rel(out[lo:lo + length].reshape(length, heads, vdim), want) < 2e-5, (step, s)
            assert rel(state[order[s]].reshape(heads, dim, vdim), held[s]) < 2e-5, (step, s)
    assert float(state[[i for i in range(slots) if i not in order]].abs().max()) == 0.0
