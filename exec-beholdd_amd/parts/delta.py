"""The gated delta rule: a matrix state per head that forgets by one factor a token and corrects what it holds under the token's key.

    q, k = Wq x, Wk x   groups x dim;   v = Wv x   heads x vdim;   head h uses q and k of group h // (heads / groups)
    q, k, v <- silu(conv(.))                              a causal convolution over time on every channel, `taps` long, no bias
    q, k <- x / sqrt(sum(x^2) + 1e-6) per head;  q <- q / sqrt(dim)
    beta = sigmoid(Wb x),  g = exp(-exp(A_log) softplus(Wa x + dt_bias))     one of each a head
    S <- g S;  S <- S + k (beta (v - S^T k))^T;  o = S^T q                   a [dim, vdim] matrix per (sequence, head), zero at the start
    out = out_scale Wo ( rms(o over each head's vdim) * w_norm * silu(Wg x) )      w_norm [vdim], the same for all heads

(The recurrence is that of S. Yang, J. Kautz, A. Hatamizadeh, "Gated Delta Networks: Improving Mamba2 with Delta Rule".)  All six
projections are one stacked product.  Per sequence the layer keeps one float32 region: the heads' states, then the last taps - 1
rows of (q, k, v) as they were projected.  The convolution's sum, the unit norms, gates, decays, the state, both of its products and the
norm are float32; the projections have the engine's activation type.  `delta_prep` makes what the recurrence reads of every row,
`delta_scan` walks a sequence's rows in order from the slot's state (prompts, portions and decode steps alike; long sequences in chunks
side by side that are joined afterwards), `gated_group_rmsnorm` norms and gates; a step of one row a sequence does all of it in one launch where the
kernel set has it (`delta_step`).  Every size and constant is a constructor parameter.
"""

from __future__ import annotations

import torch

from ..weights.binder import TensorSpec
from .base import MIXERS, CacheNeed
from .linear import Linear


class GatedDeltaRule:
    graph_safe = True      # forward reads only the step's device tensors
    graph_safe_rows = None
    writes_fresh = True    # forward(..., fresh=True) writes its result instead of adding it

    def __init__(self, hidden: int, n_heads: int, n_groups: int, dim: int, vdim: int, taps: int, norm_eps: float, prefix: str, *,
                 out_scale: float = 1.0):
        if n_heads % n_groups:
            raise ValueError(f"{n_heads} heads do not fall evenly to {n_groups} heads of queries and keys")
        if taps < 1:
            raise ValueError(f"a convolution has at least one tap, got {taps}")
        self.hidden, self.n_heads, self.n_groups, self.dim, self.vdim = int(hidden), int(n_heads), int(n_groups), int(dim), int(vdim)
        self.taps, self.norm_eps, self.prefix, self.out_scale = int(taps), float(norm_eps), prefix, float(out_scale)
        self.key_width, self.value_width = self.n_groups * self.dim, self.n_heads * self.vdim
        self.channels = 2 * self.key_width + self.value_width
        self.g_first = self.channels
        self.b_first = self.g_first + self.value_width
        self.a_first = self.b_first + self.n_heads
        self.proj = Linear(hidden, [self.key_width, self.key_width, self.value_width, self.value_width, self.n_heads, self.n_heads],
                           [prefix + name for name in ("q", "k", "v", "g", "b", "a")], whole=16)
        self.out = Linear(self.value_width, hidden, prefix + "o")
        self.state_floats = self.n_heads * self.dim * self.vdim
        self.conv_weight = self.a_log = self.dt_bias = self.norm_weight = None

    @property
    def input_reader(self):
        return self.proj.reader()

    def tensor_specs(self):
        convolutions = [TensorSpec(f"{self.prefix}{name}.conv", (width, self.taps), "linear")
                        for name, width in (("q", self.key_width), ("k", self.key_width), ("v", self.value_width))]
        return self.proj.tensor_specs() + self.out.tensor_specs() + convolutions + [
            TensorSpec(self.prefix + "A_log", (self.n_heads,), "linear"), TensorSpec(self.prefix + "dt_bias", (self.n_heads,), "linear"),
            TensorSpec(self.prefix + "norm", (self.vdim,), "norm")]

    def load(self, get):
        self.proj.load(get)
        self.out.load(get)
        f32 = lambda name: get(self.prefix + name).to(torch.float32).contiguous()
        self.conv_weight = torch.cat([f32(f"{name}.conv") for name in ("q", "k", "v")], dim=0).contiguous()
        self.a_log, self.dt_bias = f32("A_log"), f32("dt_bias")
        # one weight for all heads, laid out once per head for the kernel that norms the heads of a row side by side; the mixer's
        # factor stands in it
        self.norm_weight = (f32("norm") * self.out_scale).repeat(self.n_heads).contiguous()

    def prepare(self, kernels):
        self.proj.prepare(kernels)
        self.out.prepare(kernels)

    def cache_need(self):
        return CacheNeed(kind="state", state_shape=(self.state_floats + (self.taps - 1) * self.channels,), state_dtype=torch.float32, in_banks=True)

    def working_bytes(self, step) -> int:
        chunks = 0
        if step.sizes is not None and hasattr(step.sizes, "delta_chunk_bytes"):
            chunks = step.sizes.delta_chunk_bytes(step.seqs, step.rows, step.max_rows_per_seq, self.n_heads, self.dim, self.vdim)
        return (chunks + self.proj.working_bytes(step, step.rows) + step.matrix(step.rows, self.channels, 4)
                + step.matrix(step.rows, 4 * self.n_heads, 4) + step.matrix(step.rows, self.value_width, 4)
                + step.matrix(step.rows, self.value_width, reader=self.out.reader_for_plan(step.act_size))
                + self.out.working_bytes(step, step.rows, accumulate=True))

    def forward(self, ctx, x, hidden, cache, then_norm=None, fresh=False):
        k = ctx.kernels
        n = ctx.n_rows
        proj = self.proj.forward(ctx, x)
        gated = ctx.new_activations(n, self.value_width, reader=self.out.reader())
        sizes = (self.n_heads, self.n_groups, self.dim, self.vdim)
        rows, to = cache.state_rows(ctx)
        one_launch = getattr(k, "delta_step", None)
        if not (one_launch is not None and ctx.max_rows_per_seq == 1 and one_launch(
                proj, 0, self.g_first, self.b_first, self.a_first, self.conv_weight, cache.state, self.state_floats, self.a_log, self.dt_bias,
                rows, self.norm_weight, self.norm_eps, gated, *sizes, **to)):
            qkv, beside = ctx.new_f32(n, self.channels), ctx.new_f32(n, 4 * self.n_heads)
            k.delta_prep(proj, 0, self.b_first, self.a_first, self.conv_weight, cache.state, self.state_floats, self.a_log, self.dt_bias, ctx.row_seq,
                         ctx.seq_start, rows, qkv, beside, *sizes)
            if self.taps > 1:      # after every reader of the old state
                k.short_conv_state(proj, 0, self.channels, self.taps, cache.state, self.state_floats, ctx.seq_start, rows, **to)
            read = ctx.new_f32(n, self.value_width)
            k.delta_scan(qkv, beside, cache.state, ctx.seq_start, rows, read, *sizes, max_rows_per_seq=ctx.max_rows_per_seq, **to)
            k.gated_group_rmsnorm(read, proj, self.g_first, self.norm_weight, self.norm_eps, gated, self.n_heads, gate_after=True)
        self.out.forward(ctx, gated, out=hidden, accumulate=not fresh)
        return None


@MIXERS.register("gated_delta_rule")
def _build_gated_delta_rule(config, layer_index, prefix, shared):
    sizes = config.layers[layer_index].mixer
    return GatedDeltaRule(config.hidden, sizes.heads, sizes.kv_heads, sizes.dim, sizes.vdim, sizes.taps, config.rms_eps, prefix + "mix.")
