"""The kernels that move a state on leave it in the rows they are told to: the same numbers as in place, and what they started from untouched."""

import pytest
import torch

from test_gpu_kernels import K, dev      # noqa: F401  (K: the fixture)

pytestmark = pytest.mark.gpu

# decode steps; walks; chunks of a few and of many rows; prompts beside decoding sequences
LENGTHS = [[1, 1, 1], [1], [5, 1, 70], [130, 64, 65, 1], [700, 1, 40], [3000]]


def both(run, state, n_seqs):
    """`run(state, rows, **to)` in place, and from and to different rows."""
    slots = 2 * n_seqs + 3
    g = torch.Generator().manual_seed(n_seqs)
    order = torch.randperm(slots, generator=g).to(torch.int32)
    read, to = order[:n_seqs], order[n_seqs:2 * n_seqs]
    before = torch.randn(slots, *state, generator=g)
    here, apart = dev(before), dev(before)
    out_here, out_apart = run(here, dev(read)), run(apart, dev(read), seq_to=dev(to))
    rows = lambda x, index: x[index.long().cuda()]
    for a, b in zip(out_here, out_apart):
        assert torch.equal(a, b)
    assert torch.equal(rows(here, read), rows(apart, to)) and not torch.equal(rows(here, read), rows(dev(before), read))
    others = torch.ones(slots, dtype=torch.bool)
    others[to.long()] = False
    assert torch.equal(apart.cpu()[others], before[others])


def layout(lengths):
    starts = torch.tensor([0] + lengths).cumsum(0).to(torch.int32)
    return dev(starts), dev(torch.repeat_interleave(torch.arange(len(lengths)), torch.tensor(lengths)).to(torch.int32))


def rows(n, width, dtype=torch.bfloat16, seed=0, spread=1.0):
    return dev((spread * torch.randn(n, width, generator=torch.Generator().manual_seed(seed))).to(dtype))


@pytest.mark.parametrize("lengths", LENGTHS)
@pytest.mark.parametrize("heads,dim,vdim", [(4, 128, 128), (2, 24, 40), (16, 64, 64)])
def test_lightning(K, lengths, heads, dim, vdim):
    n, (starts, _) = sum(lengths), layout(lengths)
    proj, decay = rows(n, heads * (2 * dim + vdim)), dev(1.0 - torch.linspace(0.02, 0.2, heads))

    def run(state, slot, **to):
        out = torch.empty(n, heads * vdim, device="cuda:0")
        K.lightning_scan(proj, 0, heads * dim, 2 * heads * dim, state, decay, starts, slot, out, heads, dim, vdim, max_rows_per_seq=max(lengths), **to)
        return [out]

    both(run, (heads, dim, vdim), len(lengths))


@pytest.mark.parametrize("lengths", LENGTHS)
@pytest.mark.parametrize("heads,vdim,n_state,groups", [(8, 64, 128, 2), (4, 40, 20, 4), (3, 200, 200, 1)])      # the last: states in LDS, walked
def test_state_space(K, lengths, heads, vdim, n_state, groups):
    n, (starts, row_seq), taps = sum(lengths), layout(lengths), 4
    conv_width = heads * vdim + 2 * groups * n_state
    proj, xbc = rows(n, conv_width + heads + conv_width % 2), rows(n, conv_width, torch.float32, 1, 0.5)
    dt_bias, a_log, skip = (dev(torch.linspace(low, high, heads)) for low, high in ((-4.0, -1.0), (0.0, 2.0), (0.5, 1.0)))

    def run(state, slot, **to):
        out = torch.empty(n, heads * vdim, device="cuda:0")
        K.short_conv_state(proj, 0, conv_width, taps, state, heads * n_state * vdim, starts, slot, **to)
        K.ssm_scan(xbc, proj, conv_width, dt_bias, a_log, skip, state, 0, starts, slot, out, heads, vdim, n_state, groups, max_rows_per_seq=max(lengths), **to)
        return [out]

    both(run, (heads * n_state * vdim + (taps - 1) * conv_width,), len(lengths))


@pytest.mark.parametrize("lengths", LENGTHS)
@pytest.mark.parametrize("heads,dim", [(4, 64), (2, 32)])
def test_time_mixing_and_gated_linear_attention(K, lengths, heads, dim):
    time_mixing_and_gated_linear_attention(K, lengths, heads, dim)


# steps whose walks go two columns a thread, whole and in chunks, a column over 4, 8 and 16 lanes
@pytest.mark.parametrize("heads,dim,lengths", [(64, 64, [300, 17, 1, 64]), (260, 36, [65]), (16, 128, [1000, 5]), (8, 256, [1000, 1]), (64, 256, [66])])
def test_time_mixing_and_gated_linear_attention_in_columns(K, lengths, heads, dim):
    assert K.lib.bh_gla_in_columns(len(lengths), max(lengths), heads, dim, dim)
    time_mixing_and_gated_linear_attention(K, lengths, heads, dim)


def time_mixing_and_gated_linear_attention(K, lengths, heads, dim):
    n, (starts, row_seq), width = sum(lengths), layout(lengths), heads * dim
    proj, z, bias, bonus = rows(n, 3 * width), rows(n, width, torch.float32, 2, 0.5), dev(torch.linspace(-3.0, 0.0, width)), dev(torch.linspace(0.0, 1.0, width))
    mu, parts = dev(torch.rand(5, width, generator=torch.Generator().manual_seed(3))), [rows(n, width, seed=s) for s in (4, 5, 6)]

    def time_mixing(state, slot, **to):
        mixed = [torch.empty(n, width, dtype=torch.bfloat16, device="cuda:0") for _ in range(5)]
        out = torch.empty(n, width, device="cuda:0")
        K.token_shift(parts[0], mu, state, heads * dim * dim, row_seq, starts, slot, mixed, **to)
        K.wkv_scan(*parts, z, bias, bonus, state, 0, starts, slot, out, heads, dim, dim, max_rows_per_seq=max(lengths), **to)
        return mixed + [out]

    def gated(state, slot, **to):
        out = torch.empty(n, width, device="cuda:0")
        K.gla_scan(proj, 0, width, 2 * width, z, bias, 16.0, dim ** -0.5, state, starts, slot, out, heads, dim, dim, max_rows_per_seq=max(lengths), **to)
        return [out]

    both(time_mixing, (heads * dim * dim + width,), len(lengths))
    both(gated, (heads, dim, dim), len(lengths))


@pytest.mark.parametrize("lengths", LENGTHS)
@pytest.mark.parametrize("heads,groups,dim,vdim", [(4, 2, 64, 64), (2, 2, 128, 128), (3, 1, 40, 24)])
def test_delta_rule(K, lengths, heads, groups, dim, vdim):
    n, (starts, row_seq), taps = sum(lengths), layout(lengths), 4
    channels = 2 * groups * dim + heads * vdim
    proj = rows(n, channels + heads * vdim + 2 * heads)
    g_first, b_first, a_first = channels, channels + heads * vdim, channels + heads * vdim + heads
    conv, a_log, dt_bias = dev(0.4 * torch.randn(channels, taps, generator=torch.Generator().manual_seed(7))), dev(torch.linspace(0.0, 2.0, heads)), dev(torch.linspace(-4.0, -1.0, heads))
    sizes, at = (heads, groups, dim, vdim), heads * dim * vdim

    def in_parts(state, slot, **to):
        qkv, beside = torch.empty(n, channels, device="cuda:0"), torch.empty(n, 4 * heads, device="cuda:0")
        out = torch.empty(n, heads * vdim, device="cuda:0")
        K.delta_prep(proj, 0, b_first, a_first, conv, state, at, a_log, dt_bias, row_seq, starts, slot, qkv, beside, *sizes)
        K.short_conv_state(proj, 0, channels, taps, state, at, starts, slot, **to)
        K.delta_scan(qkv, beside, state, starts, slot, out, *sizes, max_rows_per_seq=max(lengths), **to)
        return [qkv, out]

    def in_one(state, slot, **to):
        out = torch.empty(n, heads * vdim, dtype=torch.bfloat16, device="cuda:0")
        took = K.delta_step(proj, 0, g_first, b_first, a_first, conv, state, at, a_log, dt_bias, slot, dev(torch.ones(heads * vdim)), 1e-6, out, *sizes, **to)
        assert took
        return [out]

    state = (at + (taps - 1) * channels,)
    both(in_parts, state, len(lengths))
    if max(lengths) == 1 and K.lib.bh_delta_step_takes(dim, vdim):
        both(in_one, state, len(lengths))


def test_rows_of_another_count_are_refused(K):
    from beholdd.kernels.library import KernelError
    starts, _ = layout([1, 1])
    slot = dev(torch.tensor([0, 1], dtype=torch.int32))
    with pytest.raises(KernelError):
        K.lightning_scan(rows(2, 3 * 64), 0, 64, 128, torch.zeros(4, 1, 64, 64, device="cuda:0"), dev(torch.ones(1)), starts, slot,
                         torch.empty(2, 64, device="cuda:0"), 1, 64, 64, seq_to=slot[:1])


def test_an_engine_steps_the_same_after_a_step_that_failed(K, tmp_path):
    """Gokazen's decode steps, one of which fails behind its launches, against steps none of which does."""
    import beholdd
    config = {"architecture": "Gokazen", "vocab": 120, "width": 64, "streams": 2, "logit_scale": 2.0, "norm": {"eps": 1e-5},
              "layers": [{"type": "lightning", "mixer": {"heads": 2, "dim": 16, "vdim": 24, "decay": [0.9, 0.99]}, "mlp": {"kind": "dense", "ff": 96}}] * 2}
    folder = beholdd.write_random_model(str(tmp_path), config, seed=4, dtype="bfloat16", std=0.06)
    seen = []
    for fails in (False, True):
        engine = beholdd.Engine(folder, dtype="bfloat16", max_tokens=512, device="cuda:0")
        assert any(g.banked for g in engine.cache.groups)
        slots = [engine.alloc_slot() for _ in range(3)]
        engine.step([beholdd.StepEntry(slot, [slot + 1, 2, 3], []) for slot in slots])
        rows_of = lambda token: [beholdd.StepEntry(slot, [token], [0]) for slot in slots]
        for token in (5, 6):
            engine.step(rows_of(token))
        if fails:
            replay = engine.graphs.step

            def broken(*args, **kw):
                replay(*args, **kw)
                raise RuntimeError("behind the launch")

            engine.graphs.step = broken
            with pytest.raises(RuntimeError, match="behind the launch"):
                engine.step(rows_of(7))
            engine.graphs.step = replay
        seen.append([engine.step(rows_of(token)).clone() for token in (8, 9, 10)])
    assert all(torch.equal(a, b) for a, b in zip(*seen))


# short sequences keep old inputs; steps of 128 rows and more walk down the rows
@pytest.mark.parametrize("lengths", LENGTHS + [[2, 3, 1, 4], [40, 100, 2]])
@pytest.mark.parametrize("taps", [2, 3, 4, 6])
@pytest.mark.parametrize("heads,kv_heads,dim", [(4, 2, 64), (24, 8, 128)])      # a few of a thread's channels, and all of them
def test_convolutions_leave_their_state(K, lengths, taps, heads, kv_heads, dim):
    n, (starts, row_seq) = sum(lengths), layout(lengths)
    channels = (heads + 2 * kv_heads) * dim
    u, weight = rows(n, channels + 8), dev(0.4 * torch.randn(channels, taps, generator=torch.Generator().manual_seed(1)))
    norms = [dev(torch.ones(h * dim)) for h in (heads, kv_heads)]
    position = dev(torch.cat([torch.arange(length) for length in lengths]).to(torch.int32))
    pages = [-(-length // 64) for length in lengths]
    table = torch.zeros(len(lengths), max(pages), dtype=torch.int32)
    for s, count in enumerate(pages):
        table[s, :count] = torch.arange(sum(pages[:s]), sum(pages[:s]) + count)

    def alone(state, slot, seq_to=None):
        out = torch.empty(n, channels, device="cuda:0")
        K.short_conv(u, 0, weight, None, state, 16, row_seq, starts, slot, out, silu=True, **({"seq_to": seq_to} if seq_to is not None else {}))
        if seq_to is None:
            K.short_conv_state(u, 0, channels, taps, state, 16, starts, slot)
        else:      # (sixteen floats that somebody else leaves)
            state[seq_to.long(), :16] = state[slot.long(), :16]
        return [out]

    def with_heads(state, slot, seq_to=None):
        q = torch.empty(n, heads * dim, dtype=torch.bfloat16, device="cuda:0")
        keys, values = (torch.zeros(shape, dtype=torch.bfloat16, device="cuda:0") for shape in ((sum(pages), kv_heads, 64, dim), (sum(pages), kv_heads, dim, 64)))
        K.conv_norm_rope_write(u, 0, weight, state, 16, starts, slot, *norms, 1e-6, None, 0, position, row_seq, q, keys, values, dev(table), heads, kv_heads, dim,
                               dim, dim, True, **({"seq_to": seq_to} if seq_to is not None else {}))
        if seq_to is None:
            K.short_conv_state(u, 0, channels, taps, state, 16, starts, slot)
        else:
            state[seq_to.long(), :16] = state[slot.long(), :16]
        return [q, keys, values]

    both(alone, (16 + (taps - 1) * channels,), len(lengths))
    both(with_heads, (16 + (taps - 1) * channels,), len(lengths))
