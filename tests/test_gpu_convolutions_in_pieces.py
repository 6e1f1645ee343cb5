"""Short convolutions over steps of many rows, in pieces of four channels and where these do not go, against plain sums in 64 bits; the
state that a step leaves is exact."""

import numpy as np
import pytest
import torch

import plain_pudorax
from test_gpu_pudorax import dev, ragged, rel, rounded

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16]


@pytest.fixture(scope="module")
def K():
    from beholdd.kernels import HipKernels
    return HipKernels("cuda:0")


# rows: stretches of sixteen that end early, and in which one or several sequences start; channels: one piece, pieces that leave lanes idle, more
# than a workgroup's; `first` and `stride` of whole pieces, and of some that are not (the walk of single channels)
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("lengths", [[128], [15, 1, 2, 160], [70, 16, 43], [130, 1]])
@pytest.mark.parametrize("channels,taps,first,stride", [(4, 4, 8, 16), (300, 3, 4, 312), (1100, 2, 0, 1100), (1032, 4, 4, 1040), (64, 4, 2, 72), (64, 4, 4, 70)])
def test_convolutions_in_pieces(K, dtype, lengths, channels, taps, first, stride):
    rng = np.random.default_rng(channels + taps + sum(lengths))
    n, n_seqs = sum(lengths), len(lengths)
    w, b = rng.standard_normal((channels, taps)).astype(np.float32), rng.standard_normal(channels).astype(np.float32)
    rows = [int(i) for i in rng.permutation(2 * n_seqs)]      # of the state: those read, then those written
    seq_start, seq_slot, row_seq, starts = ragged(lengths, rows[:n_seqs])
    before = rng.standard_normal((2 * n_seqs, (taps - 1) * channels)).astype(np.float32)
    u_t, u = rounded(rng.standard_normal((n, stride)), dtype)
    state, out = dev(before), torch.empty(n, channels, device="cuda:0")
    K.short_conv(dev(u_t), first, dev(w), dev(b), state, 0, row_seq, seq_start, seq_slot, out, silu=True, seq_to=dev(np.array(rows[n_seqs:], np.int32)))
    for s, length in enumerate(lengths):
        lo = starts[s]
        inputs = np.concatenate([before[rows[s]].reshape(taps - 1, channels), u[lo:lo + length, first:first + channels]])
        want = plain_pudorax.silu(plain_pudorax.short_conv(inputs, w, b))[taps - 1:]
        assert rel(out[lo:lo + length], want) < 1e-5, s
        assert np.array_equal(state[rows[n_seqs + s]].cpu().numpy().reshape(taps - 1, channels), inputs[-(taps - 1):].astype(np.float32)), s
        assert np.array_equal(state[rows[s]].cpu().numpy(), before[rows[s]])
