"""Time mixing in the manner of RWKV: a matrix state per head whose rows decay each by a factor that the token sets, read before the
token is written into it, and a bonus with which a token reads itself.

    z_s = h + (h' - h) mu_s   for s in r, k, v, g, w;  h' is the token before's h (zeros ahead of the first)
    r, k, v = W_s z_s                                       heads x dim
    a = exp(-exp(W_w2 tanh(W_w1 z_w) + w0))                 heads x dim, one decay per key channel, through a low rank
    o_t = (S_(t-1) + diag(u) k_t v_t^T)^T r_t               u [heads, dim]
    S_t = diag(a_t) S_(t-1) + k_t v_t^T                     a [dim, dim] matrix per (sequence, head), zero at the start
    out = Wo ( rms(o_t over each head's dim) * w_norm * silu(W_g z_g) )      w_norm [heads * dim]

(The recurrence is that of B. Peng et al., "Eagle and Finch: RWKV with Matrix-Valued States and Dynamic Recurrence".)  Per sequence the
layer keeps one float32 region: the heads' states, then the last token's h.  The mixes and the projections have the engine's activation
type; the decays with their tanh and exponentials, the bonus, the state, its products and the norm are float32.  `token_shift` makes the
five mixes of a step's rows and moves the kept h on, `wkv_scan` walks a sequence's rows in order from the slot's state (prompts, portions and
decode steps alike; long sequences in chunks side by side), `gated_group_rmsnorm` norms the heads and gates.  Every size and constant is a
constructor parameter.
"""

from __future__ import annotations

import torch

from ..weights.binder import TensorSpec
from .base import MIXERS, CacheNeed
from .linear import Linear


class TimeMixing:
    graph_safe = True      # forward reads only the step's device tensors
    graph_safe_rows = None
    writes_fresh = True    # forward(..., fresh=True) writes its result instead of adding it
    MIXES = ("r", "k", "v", "g", "w")

    def __init__(self, hidden: int, n_heads: int, dim: int, decay_rank: int, norm_eps: float, prefix: str):
        self.hidden, self.n_heads, self.dim, self.decay_rank = int(hidden), int(n_heads), int(dim), int(decay_rank)
        self.norm_eps, self.prefix, self.width = float(norm_eps), prefix, int(n_heads) * int(dim)
        self.projections = {name: Linear(hidden, self.width, prefix + name) for name in ("r", "k", "v", "g")}
        # (a whole tile of outputs, with rows of zeros behind the rank's: a product of many rows then cuts K into parts)
        self.decay_down = Linear(hidden, self.decay_rank, prefix + "w1", whole=128)
        self.decay_up = Linear(self.decay_rank, self.width, prefix + "w2")
        self.out = Linear(self.width, hidden, prefix + "o")
        self.state_floats = self.n_heads * self.dim * self.dim
        self.mu = self.decay_bias = self.bonus = self.norm_weight = None

    def _linears(self):
        return [*self.projections.values(), self.decay_down, self.decay_up, self.out]

    def tensor_specs(self):
        specs = [spec for linear in self._linears() for spec in linear.tensor_specs()]
        specs += [TensorSpec(f"{self.prefix}mu.{name}", (self.hidden,), "linear") for name in self.MIXES]
        return specs + [TensorSpec(self.prefix + "w0", (self.width,), "linear"), TensorSpec(self.prefix + "u", (self.n_heads, self.dim), "linear"),
                        TensorSpec(self.prefix + "norm", (self.width,), "norm")]

    def load(self, get):
        for linear in self._linears():
            linear.load(get)
        f32 = lambda name: get(self.prefix + name).to(torch.float32).contiguous()
        self.mu = torch.stack([f32(f"mu.{name}") for name in self.MIXES]).contiguous()
        self.decay_bias, self.bonus, self.norm_weight = f32("w0"), f32("u").reshape(-1).contiguous(), f32("norm")

    def prepare(self, kernels):
        for linear in self._linears():
            linear.prepare(kernels)

    def cache_need(self):
        return CacheNeed(kind="state", state_shape=(self.state_floats + self.hidden,), state_dtype=torch.float32, in_banks=True)

    def working_bytes(self, step) -> int:
        chunks = 0
        if step.sizes is not None and hasattr(step.sizes, "gla_chunk_bytes"):
            chunks = step.sizes.gla_chunk_bytes(step.seqs, step.rows, step.max_rows_per_seq, self.n_heads, self.dim, self.dim)
        mixes = len(self.MIXES) * step.matrix(step.rows, self.hidden, reader=self.projections["r"].reader_for_plan(step.act_size))
        return (chunks + mixes + sum(linear.working_bytes(step, step.rows) for linear in self.projections.values())
                + self.decay_down.working_bytes(step, step.rows, out_size=4) + step.matrix(step.rows, self.decay_rank)
                + self.decay_up.working_bytes(step, step.rows, out_size=4) + step.matrix(step.rows, self.width, 4)
                + step.matrix(step.rows, self.width, reader=self.out.reader_for_plan(step.act_size))
                + self.out.working_bytes(step, step.rows, accumulate=True))

    def forward(self, ctx, x, hidden, cache, then_norm=None, fresh=False):
        k = ctx.kernels
        n = ctx.n_rows
        reader = self.projections["r"].reader()
        mixed = {name: ctx.new_activations(n, self.hidden, reader=reader) for name in self.MIXES}
        rows, to = cache.state_rows(ctx)
        k.token_shift(x, self.mu, cache.state, self.state_floats, ctx.row_seq, ctx.seq_start, rows, [mixed[name] for name in self.MIXES], **to)
        projected = {name: linear.forward(ctx, mixed[name]) for name, linear in self.projections.items()}
        low = self.decay_down.forward(ctx, mixed["w"], out_dtype=torch.float32)
        bent = ctx.new_activations(n, self.decay_rank, reader=self.decay_up.reader())
        k.tanh_rows(low, bent)
        decays = self.decay_up.forward(ctx, bent, out_dtype=torch.float32)
        read = ctx.new_f32(n, self.width)
        k.wkv_scan(projected["r"], projected["k"], projected["v"], decays, self.decay_bias, self.bonus, cache.state, 0, ctx.seq_start, rows,
                   read, self.n_heads, self.dim, self.dim, max_rows_per_seq=ctx.max_rows_per_seq, **to)
        gated = ctx.new_activations(n, self.width, reader=self.out.reader())
        k.gated_group_rmsnorm(read, projected["g"], 0, self.norm_weight, self.norm_eps, gated, self.n_heads, gate_after=True)
        self.out.forward(ctx, gated, out=hidden, accumulate=not fresh)
        return None


@MIXERS.register("time_mixing")
def _build_time_mixing(config, layer_index, prefix, shared):
    sizes = config.layers[layer_index].mixer
    return TimeMixing(config.hidden, sizes.heads, sizes.dim, sizes.decay_rank, config.rms_eps, prefix + "mix.")
