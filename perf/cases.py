"""What a user of this framework has it do on a GPU, as cases whose time is worth measuring.

A case is one of three calls of the public interface on a model with random weights that is made from a configuration:

  prefill    whole prompts of new sequences through one `Engine.step`, logits of the last `want` positions of each (1: the first
             token of an answer; more: the positions of an answer whose likelihood is asked for)
  decode     one more token for every live sequence, whose prompts are in the cache, through `Engine.step`; the tokens are given
  generate   `Engine.generate` from prompts to answers, with the logits that every token is chosen from

The architectures are Qwen3 (the framework's first one) and three of the others, which between them hold one of each kind of mixer
and feed-forward: Gokazen (linear attention with a decay, attention over a cached latent, residual streams), Pudorax (convolved and
gated attention, a state-space recurrence, routed experts) and Vitudra (time mixing, the gated delta rule beside chunk attention,
attention with a distance bias).  Layer sizes are those of `bench.py`: widths of 1,024 to 5,120, heads of 128, a vocabulary of
32,768, and 2 to 8 of a model's layers, so that three of them are made quickly.

`exact` says what the logits are in 64-bit arithmetic, for whole sequences, without this package's code.
"""

import hashlib
import math

import numpy as np
import torch

import beholdd

DEVICE = "cuda:0"
VOCAB = 32768
NEW_TOKENS = 4096      # a decode case's sequences may grow by so many tokens; then they start again from their prompts
ROWS_PER_STEP = 8192   # prompts of a decode case go into the cache in steps of at most so many tokens


# ---- the cases ----------------------------------------------------------------------------------------------------

def listed():
    return [
        # One user's conversation with a small model: nothing but launches and latency.
        dict(name="qwen3_decode_1", do="decode", arch="Qwen3", dtype="bfloat16", width=1024, kv_ratio=2, layers=8, ff=3072, batch=1, shortest=1500, longest=1500),
        # The headline: eight sequences at the end of a context of 8,192 tokens.
        dict(name="qwen3_decode_8_long", do="decode", arch="Qwen3", dtype="bfloat16", width=4096, kv_ratio=4, layers=8, ff=12288, batch=8, shortest=7900, longest=8100),
        # A server with many short conversations of unequal lengths.
        dict(name="qwen3_decode_64", do="decode", arch="Qwen3", dtype="bfloat16", width=4096, kv_ratio=4, layers=8, ff=12288, batch=64, shortest=256, longest=1024),
        # A few short questions that arrive together: too few rows to fill the chip, and not a multiple of anything.
        dict(name="qwen3_prefill_short", do="prefill", arch="Qwen3", dtype="bfloat16", width=5120, kv_ratio=5, layers=4, ff=17408, batch=3, shortest=37, longest=131, want=1),
        # Long documents: the largest step there is in ordinary use.
        dict(name="qwen3_prefill_4x2048", do="prefill", arch="Qwen3", dtype="bfloat16", width=4096, kv_ratio=4, layers=8, ff=12288, batch=4, shortest=1900, longest=2180, want=1),
        # Answers from the 32-bit engine, as somebody takes them who checks a model or compares log-probabilities.
        dict(name="qwen3_float32_generate", do="generate", arch="Qwen3", dtype="float32", width=1024, kv_ratio=2, layers=8, ff=3072, batch=4, shortest=40, longest=300, new=16,
             temperature=0.0, top_k=0, top_p=1.0),
        # The other architectures, each with a prompt and with a batch that is decoded.
        dict(name="gokazen_prefill_2048", do="prefill", arch="Gokazen", dtype="bfloat16", width=2048, layers=8, batch=1, shortest=2048, longest=2048, want=1),
        dict(name="gokazen_decode_16", do="decode", arch="Gokazen", dtype="bfloat16", width=4096, layers=8, batch=16, shortest=500, longest=4000),
        dict(name="pudorax_prefill_3", do="prefill", arch="Pudorax", dtype="bfloat16", width=2048, layers=3, batch=3, shortest=300, longest=1100, want=64),
        dict(name="pudorax_decode_16", do="decode", arch="Pudorax", dtype="bfloat16", width=2048, layers=3, batch=16, shortest=1000, longest=2000),
        dict(name="vitudra_prefill_2048", do="prefill", arch="Vitudra", dtype="bfloat16", width=4096, layers=4, batch=1, shortest=2048, longest=2048, want=16),
        dict(name="vitudra_decode_8", do="decode", arch="Vitudra", dtype="bfloat16", width=2048, layers=8, batch=8, shortest=1000, longest=4000),
    ]


def _between(rng, low, high):
    """A whole number from low to high, spread over its logarithm."""
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    arch = rng.choice(["Qwen3", "Qwen3", "Qwen3", "Gokazen", "Pudorax", "Vitudra"])
    do = rng.choice(["prefill", "decode", "generate"] if arch == "Qwen3" else ["prefill", "decode"])
    case = dict(do=do, arch=arch, dtype="float32" if do == "generate" else "bfloat16")
    if arch == "Qwen3":
        case["width"] = rng.choice([1024, 2048] if do == "generate" else [1024, 2048, 2560, 4096, 5120])
        case["kv_ratio"] = rng.choice({5120: [5, 8], 2560: [4, 5]}.get(case["width"], [2, 4, 8]))
        case["layers"] = rng.randint(2, 4 if case["width"] == 5120 else 8)
        case["ff"] = 128 * rng.randint(case["width"] * 5 // 256, case["width"] * 7 // 256)
    else:
        case["width"] = rng.choice([1024, 2048, 4096] if arch != "Pudorax" else [1024, 2048])
        case["layers"] = {"Gokazen": 4 * rng.randint(1, 2), "Pudorax": 3, "Vitudra": 4 * rng.randint(1, 2)}[arch]
    if do == "prefill":
        case["batch"] = _between(rng, 1, 8)
        case["longest"] = _between(rng, 16, min(4096, 8192 // case["batch"] if arch == "Qwen3" else 4096 // case["batch"]))
        case["want"] = min(64 if arch == "Pudorax" else rng.choice([1, 1, 16]), case["longest"])
    elif do == "decode":
        case["batch"] = _between(rng, 1, 64)
        case["longest"] = _between(rng, 100, min(8100, 65536 // case["batch"] if arch == "Qwen3" else 32768 // case["batch"]))
    else:
        case["batch"], case["longest"] = _between(rng, 1, 8), _between(rng, 16, 400)
        case["new"] = rng.randint(4, 16)
        sampling = rng.choice([dict(temperature=0.0, top_k=0, top_p=1.0), dict(temperature=1.0, top_k=0, top_p=1.0),
                               dict(temperature=0.8, top_k=50, top_p=0.9)])
        case.update(sampling)
    case["shortest"] = max(min(case.get("want", 1), case["longest"]), case["longest"] // rng.choice([1, 2, 5]))
    return case


# ---- configurations -----------------------------------------------------------------------------------------------

def config_of(case):
    """The configuration file's content for a case's model."""
    width, layers, heads = case["width"], case["layers"], case["width"] // 128
    if case["arch"] == "Qwen3":
        return {"architectures": ["Qwen3ForCausalLM"], "model_type": "qwen3", "num_hidden_layers": layers, "hidden_size": width,
                "num_attention_heads": heads, "num_key_value_heads": heads // case["kv_ratio"], "head_dim": 128,
                "intermediate_size": case["ff"], "vocab_size": VOCAB, "rope_theta": 1000000.0, "rms_norm_eps": 1e-6,
                "max_position_embeddings": 40960, "tie_word_embeddings": False}
    if case["arch"] == "Gokazen":      # three layers with linear attention to every one with attention over a latent
        mlp = {"kind": "dense", "ff": 3 * width}
        decay = [1.0 - 2.0 ** (-5.0 - 3.0 * h / max(heads - 1, 1)) for h in range(heads)]
        lightning = {"type": "lightning", "mixer": {"heads": heads, "dim": 128, "vdim": 128, "decay": decay}, "mlp": mlp}
        latent = {"type": "latent_attention", "mlp": mlp,
                  "mixer": {"heads": heads, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 192, "scale": 192 ** -0.5,
                            "rot": {"base": 10000.0, "dims": 64}}}
        return {"architecture": "Gokazen", "vocab": VOCAB, "width": width, "streams": 2, "logit_scale": 1.0,
                "norm": {"eps": 1e-6}, "layers": [latent if i % 4 == 3 else lightning for i in range(layers)]}
    if case["arch"] == "Pudorax":      # three layers of which one runs twice; 32 experts of which 4 are used, and a shared one
        mlp = {"kind": "moe", "router": {"experts": 32, "top": 4}, "expert": {"ff": 3 * width // 8, "limit": 7.0},
               "shared": {"ff": 3 * width // 2, "limit": 7.0}}
        attention = {"type": "attention", "mlp": mlp,
                     "mixer": {"heads": heads, "kv_heads": max(heads // 4, 1), "dim": 128, "vdim": 128, "conv": 4,
                               "scale": 128 ** -0.5, "rot": {"base": 1000000.0, "dims": 64}}}
        mamba = {"type": "mamba2", "mlp": mlp,
                 "mixer": {"heads": 2 * width // 64, "vdim": 64, "state": 128, "groups": 8, "norm_groups": 8, "conv": 4}}
        return {"architecture": "Pudorax", "vocab": VOCAB, "width": width, "embedding": {"scale": 1.0}, "logit_softcap": 30.0,
                "norm": {"eps": 1e-6}, "token_side": {"dim": 256}, "loop": {"start": 1, "stop": 2, "times": 2},
                "layers": [attention, mamba, attention]}
    if case["arch"] == "Vitudra":
        span, mlp = 4096, {"kind": "dense", "ff": 3 * width}
        heads_of = {"heads": heads, "kv_heads": max(heads // 4, 1), "dim": 128, "vdim": 128, "scale": 128 ** -0.5,
                    "mask": {"size": span}}
        left = dict(heads_of, softcap=50.0, rot={"base": 1000000.0, "dims": 64, "scaling": {"factor": 8.0}})
        right = {"heads": heads, "kv_heads": heads // 2, "dim": 128, "vdim": 128, "conv": 4}
        q_temp = {"coef": 0.1, "every": 8192}
        kinds = []
        for first in range(0, layers, 4):
            kinds += [{"type": "parallel", "mixer": {"left": left, "right": right, "left_scale": 0.7, "right_scale": 0.7}, "mlp": mlp},
                      {"type": "attention", "mixer": dict(heads_of, q_temp=q_temp), "mlp": mlp},
                      {"type": "wkv", "mixer": {"heads": width // 64, "dim": 64, "decay_rank": 64}, "mlp": mlp},
                      {"type": "attention", "mixer": dict(heads_of, q_temp=q_temp, kv_from=first + 1), "mlp": mlp}]
        return {"architecture": "Vitudra", "vocab": VOCAB, "width": width, "norm": {"eps": 1e-6}, "residual_mult": 0.3, "layers": kinds}
    raise ValueError(case["arch"])


# ---- weights and tokens, from the seed alone ----------------------------------------------------------------------

def _key(seed, *what):
    return int.from_bytes(hashlib.sha256(repr((int(seed),) + what).encode()).digest()[:7], "little")


def weight(case, seed, name, shape):
    """One tensor: N(0, 0.02) for matrices; around 1 for scales (around 0 where the design stores w of 1 + w); convolutions, decays
    and token mixes spread as trained models have them, and routers that mean their first choices (the last of the chosen experts
    weighs little, as does a close call between it and the next one), experts that add little to the residual."""
    dtype = torch.bfloat16 if case["dtype"] == "bfloat16" else torch.float32
    generator = torch.Generator(device=DEVICE)
    generator.manual_seed(_key(seed, name))
    last = name.rsplit(".", 1)[-1]
    uniform = {"A_log": (0.0, 2.0), "dt_bias": (-5.0, -1.0), "w0": (-6.0, -1.0)}.get(last)
    if ".mu." in name:
        uniform = (0.0, 1.0)
    out = torch.empty(tuple(shape), dtype=dtype, device=DEVICE)
    if uniform is not None:
        return out.uniform_(*uniform, generator=generator)
    spread = 0.4 if last == "conv" or name.endswith(".mix.u") else 0.12 if last == "router" else 0.01 if ".mlp.e" in name and last == "down" else 0.02
    out.normal_(0.0, spread, generator=generator)
    if last == "mix" and ".hc" in name:
        return out + torch.eye(shape[0], dtype=dtype, device=DEVICE)
    scale = (last in ("norm1", "norm2", "norm", "ls1", "ls2", "D", "in", "out") and len(shape) == 1) or name.endswith("norm.weight")
    around_zero = case["arch"] in ("Gokazen", "Vitudra") and (last in ("norm1", "norm2") or name == "final.norm")
    return out + 1.0 if scale and not around_zero else out


def _numbers(case, seed):
    return np.random.default_rng(_key(seed, "inputs"))


def _lengths(case, numbers):
    return [int(n) for n in numbers.integers(case["shortest"], case["longest"] + 1, case["batch"])]


def _prompts(case, seed):
    numbers = _numbers(case, seed)
    lengths = _lengths(case, numbers)
    return [numbers.integers(0, VOCAB, n).tolist() for n in lengths]


def _given(case, seed):
    """A decode case's tokens: [step][sequence]."""
    return np.random.default_rng(_key(seed, "given")).integers(0, VOCAB, (NEW_TOKENS, case["batch"])).tolist()


# ---- what is measured ---------------------------------------------------------------------------------------------

def prepare(case, seed):
    config = config_of(case)
    architecture = beholdd.resolve_architecture(config)
    model = architecture.build(architecture.config_class.from_dict(config))
    shapes = {spec.name: spec.shape for spec in model.tensor_specs()}
    model.load(lambda name: weight(case, seed, name, shapes[name]), torch.device(DEVICE))
    prompts = _prompts(case, seed)
    more = {"prefill": 0, "decode": NEW_TOKENS, "generate": case.get("new", 0)}[case["do"]]
    room = sum(-(-(len(p) + more) // 64) * 64 for p in prompts)
    engine = beholdd.Engine(model=model, dtype=case["dtype"], max_tokens=room, max_slots=len(prompts), device=DEVICE)
    state = {"case": case, "engine": engine, "prompts": prompts, "seed": seed}
    if case["do"] == "decode":
        state["given"] = _given(case, seed)
        _start(state)
    return state


def _start(state):
    """A decode case's sequences, their prompts in the cache."""
    engine, prompts = state["engine"], state["prompts"]
    for slot in state.get("slots", ()):
        engine.free_slot(slot)
    state["slots"] = slots = [engine.alloc_slot() for _ in prompts]
    state["step"] = 0
    entries, rows = [], 0
    for slot, prompt in zip(slots, prompts):
        if rows + len(prompt) > ROWS_PER_STEP and entries:
            engine.step(entries)
            entries, rows = [], 0
        entries.append(beholdd.StepEntry(slot, prompt, []))
        rows += len(prompt)
    engine.step(entries)


def run(state):
    engine, case = state["engine"], state["case"]
    if case["do"] == "prefill":
        slots = [engine.alloc_slot() for _ in state["prompts"]]
        logits = engine.step([beholdd.StepEntry(slot, prompt, list(range(len(prompt) - case["want"], len(prompt))))
                              for slot, prompt in zip(slots, state["prompts"])])
        for slot in slots:
            engine.free_slot(slot)
        return logits
    if case["do"] == "decode":
        if state["step"] == NEW_TOKENS:
            _start(state)
        tokens = state["given"][state["step"]]
        state["step"] += 1
        return engine.step([beholdd.StepEntry(slot, [token], [0]) for slot, token in zip(state["slots"], tokens)])
    logits = [[] for _ in state["prompts"]]
    results = engine.generate(state["prompts"], max_new_tokens=case["new"], temperature=case["temperature"], top_k=case["top_k"],
                              top_p=case["top_p"], seed=state["seed"] % 65536,
                              on_logits=lambda index, step, row: logits[index].append(row.clone()))
    return {"logits": torch.stack([torch.stack(rows) for rows in logits]),
            "tokens": torch.tensor([result.token_ids for result in results])}


def tolerance(case):
    # float32: sums of 1,024 to 7,168 products in another order, 1.0e-6 to 1.6e-6 away from 64 bits.  bfloat16: every sublayer's
    # operands rounded to 8 bits, 0.007 to 0.017 away from 64 bits (the upper end where a router's close calls go the other way).
    if case["dtype"] == "float32":
        return {"rel": 1e-5, "max": 2e-4, "differ": 0.0}
    return {"rel": 0.03, "max": 0.4}


# ---- what a pass cannot do without --------------------------------------------------------------------------------

def _layer_work(case, layer, rows):
    """(weights read, multiplications a row, cached numbers of a position, state numbers of a sequence, flops a row and seen position) of a layer run."""
    width, heads = case["width"], case["width"] // 128
    if case["arch"] == "Qwen3":
        kv = heads // case["kv_ratio"] * 128
        weights = width * (2 * width + 2 * kv) + 3 * width * case["ff"]
        return weights, weights, 2 * kv, 0, 4 * width
    m = layer["mixer"]
    if case["arch"] == "Gokazen":
        ff = 2 * width * 3 * width
        if layer["type"] == "lightning":
            return 5 * width * width + ff, 5 * width * width + ff + 2 * heads * 128 * 128, 0, heads * 128 * 128, 0
        weights = width * (heads * 192 + 256 + width) + 2 * width * 192 + ff
        return weights, weights, 256, 0, heads * (2 * 256 + 2 * 192)
    if case["arch"] == "Pudorax":
        expert = 3 * width * (3 * width // 8)
        read = 3 * width * (3 * width // 2) + width * 32 + expert * 32 * (1.0 - (1.0 - 4 / 32) ** rows) + 2 * width * 256
        used = 3 * width * (3 * width // 2) + width * 32 + expert * 4 + 2 * width * 256
        if layer["type"] == "attention":
            kv = m["kv_heads"] * 128
            own = width * (3 * width + 2 * kv)
            return own + read, own + used, 2 * kv, 3 * (width + 2 * kv), 4 * width
        inner = 2 * width
        own = width * (2 * inner + 2 * 8 * 128 + m["heads"]) + inner * width
        return own + read, own + used + 3 * inner * 128, 0, inner * 128, 0
    ff, kv = 9 * width * width, max(heads // 4, 1) * 128
    if layer["type"] == "attention":
        own = 2 * width * width + (0 if "kv_from" in m else 2 * width * kv) + ff
        return own, own, 2 * kv, 0, 4 * width
    if layer["type"] == "wkv":
        own = 5 * width * width + 128 * width + ff
        return own, own + 3 * width * 64, 0, width * 64, 0
    own = 2 * width * width + 2 * width * kv + width * (2 * width + 2 * (width // 2)) + 2 * width * heads + ff
    return own, own + 4 * width * 128, 2 * kv, width * 128 + 3 * 2 * width, 4 * width


def _runs(config):
    layers, loop = config.get("layers"), config.get("loop")
    if layers is None:
        return [None] * config["num_hidden_layers"]
    if not loop:
        return layers
    return layers[:loop["start"]] + layers[loop["start"]:loop["stop"]] * loop["times"] + layers[loop["stop"]:]


def work(case):
    config, size = config_of(case), 2 if case["dtype"] == "bfloat16" else 4
    mean = (case["shortest"] + case["longest"]) / 2
    head = VOCAB * case["width"]

    def step(rows, new, past, wanted):
        """`batch` sequences bring `new` tokens each to `past`."""
        moved = size * (head + rows * case["width"]) + 4 * wanted * VOCAB
        flops = 2 * head * wanted
        for layer in _runs(config):
            weights, products, cached, state, seen = _layer_work(case, layer, rows)
            moved += size * (weights + case["batch"] * cached * (past + new)) + 4 * case["batch"] * state * (2 if past else 1)
            flops += rows * (2 * products + seen * (past + (new + 1) / 2))
        if config.get("loop"):
            moved += size * 2 * case["width"] ** 2
            flops += rows * 4 * case["width"] ** 2 * config["loop"]["times"]
        return moved, flops

    batch = case["batch"]
    if case["do"] == "decode":
        steps = [step(batch, 1, mean, batch)]
    elif case["do"] == "prefill":
        steps = [step(batch * mean, mean, 0, batch * case["want"])]
    else:
        steps = [step(batch * mean, mean, 0, batch)] + [step(batch, 1, mean + i, batch) for i in range(1, case["new"])]
    return {"bytes": sum(s[0] for s in steps), "flops": sum(s[1] for s in steps)}


# ---- the same in 64 bits ------------------------------------------------------------------------------------------
# Whole sequences side by side, filled up to the longest behind their ends: every architecture here is causal, so what stands
# behind a position does not reach it.  x: [sequences, positions, width].

class _Weights:
    def __init__(self, case, seed):
        self.case, self.seed = case, seed

    def __call__(self, name, *shape):
        return weight(self.case, self.seed, name, shape).double()


def _linear(x, w):
    return x @ w.T


def _rms(x, eps=1e-6):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _angles(t_len, dims, base, factor=1.0):
    """Position times frequency, a float32 product of float32 numbers by the designs' definition."""
    freqs = torch.tensor([base ** (-2.0 * i / dims) / factor for i in range(dims // 2)], dtype=torch.float64).float()
    return (torch.arange(t_len).float()[:, None] * freqs[None, :]).double().to(DEVICE)


def _turn(x, angles, pairs):
    """The first dims of x [B, T, heads, n] turned: neighbours (2i, 2i + 1) or halves (i, i + dims / 2)."""
    dims = 2 * angles.shape[1]
    cos, sin = angles.cos()[:, None, :], angles.sin()[:, None, :]
    first, second = (slice(0, dims, 2), slice(1, dims, 2)) if pairs else (slice(0, dims // 2), slice(dims // 2, dims))
    out = x.clone()
    out[..., first] = x[..., first] * cos - x[..., second] * sin
    out[..., second] = x[..., second] * cos + x[..., first] * sin
    return out


def _attend(q, k, v, scale, window=0, chunk=0, cap=0.0, slopes=None):
    """Causal softmax attention: q [B, T, H, d], k [B, T, G, d], v [B, T, G, e] -> [B, T, H * e]."""
    batch, t_len, heads, _ = q.shape
    per = heads // k.shape[2]
    out = torch.empty(batch, t_len, heads, v.shape[3], dtype=torch.float64, device=DEVICE)
    at = torch.arange(t_len, device=DEVICE)
    distance = at[:, None] - at[None, :]
    hidden = distance < 0
    if window:
        hidden |= distance >= window
    if chunk:
        hidden |= (at[:, None] // chunk) != (at[None, :] // chunk)
    for b in range(batch):
        for head in range(heads):
            scores = (q[b, :, head] @ k[b, :, head // per].T).mul_(scale)
            if cap:
                scores = torch.tanh(scores / cap) * cap
            if slopes is not None:
                scores -= slopes[head] * distance
            scores.masked_fill_(hidden, -math.inf)
            out[b, :, head] = torch.softmax(scores, -1) @ v[b, :, head // per]
    return out.reshape(batch, t_len, -1)


def _heads(x, n):
    return x.reshape(x.shape[0], x.shape[1], n, -1)


def _conv(x, taps):
    """Causal filter over time of x [B, T, C] with taps [C, n], the last on the present."""
    n = taps.shape[1]
    padded = torch.nn.functional.pad(x, (0, 0, n - 1, 0))
    return sum(padded[:, j:j + x.shape[1]] * taps[:, j] for j in range(n))


def _silu(x):
    return x * torch.sigmoid(x)


def _qwen3(case, w, tokens, wanted):
    c = config_of(case)
    width, heads, groups, ff = case["width"], c["num_attention_heads"], c["num_key_value_heads"], case["ff"]
    angles = _angles(tokens.shape[1], 128, c["rope_theta"])
    x = w("model.embed_tokens.weight", VOCAB, width)[tokens]
    for i in range(case["layers"]):
        p = f"model.layers.{i}."
        h = _rms(x) * w(p + "input_layernorm.weight", width)
        q = _heads(_linear(h, w(p + "self_attn.q_proj.weight", width, width)), heads)
        k = _heads(_linear(h, w(p + "self_attn.k_proj.weight", groups * 128, width)), groups)
        v = _heads(_linear(h, w(p + "self_attn.v_proj.weight", groups * 128, width)), groups)
        q = _turn(_rms(q) * w(p + "self_attn.q_norm.weight", 128), angles, False)
        k = _turn(_rms(k) * w(p + "self_attn.k_norm.weight", 128), angles, False)
        x = x + _linear(_attend(q, k, v, 128 ** -0.5), w(p + "self_attn.o_proj.weight", width, width))
        h = _rms(x) * w(p + "post_attention_layernorm.weight", width)
        gated = _silu(_linear(h, w(p + "mlp.gate_proj.weight", ff, width))) * _linear(h, w(p + "mlp.up_proj.weight", ff, width))
        x = x + _linear(gated, w(p + "mlp.down_proj.weight", width, ff))
    return _linear(_rms(wanted(x)) * w("model.norm.weight", width), w("lm_head.weight", VOCAB, width))


def _lightning(h, w, p, m, width):
    heads = m["heads"]
    q, k, v = (_heads(_silu(_linear(h, w(p + s, heads * 128, width))), heads) for s in "qkv")
    decay = torch.tensor(m["decay"], dtype=torch.float64, device=DEVICE).float().double()[None, :, None, None]
    state = torch.zeros(h.shape[0], heads, 128, 128, dtype=torch.float64, device=DEVICE)
    o = torch.empty_like(v)
    for t in range(h.shape[1]):
        state = decay * state + k[:, t, :, :, None] * v[:, t, :, None, :]
        o[:, t] = (q[:, t, :, None, :] @ state)[:, :, 0]
    o = _rms(o.reshape(h.shape)) * w(p + "norm", heads * 128) * torch.sigmoid(_linear(h, w(p + "g", heads * 128, width)))
    return _linear(o, w(p + "o", width, heads * 128))


def _latent(h, w, p, m, width):
    heads, rank, rot = m["heads"], m["kv_rank"], m["rot_dim"]
    angles = _angles(h.shape[1], rot, m["rot"]["base"])
    q = _heads(_linear(h, w(p + "q", heads * (128 + rot), width)), heads)
    down = _linear(h, w(p + "dkv", rank + rot, width))
    latent = _rms(down[..., :rank]) * w(p + "dkv.norm", rank)
    k = _heads(_linear(latent, w(p + "uk", heads * 128, rank)), heads)
    v = _heads(_linear(latent, w(p + "uv", heads * 128, rank)), heads)
    turned = _turn(down[:, :, None, rank:], angles, False).expand(-1, -1, heads, -1)
    o = _attend(torch.cat([q[..., :128], _turn(q[..., 128:], angles, False)], -1), torch.cat([k, turned], -1), v, m["scale"])
    return _linear(o, w(p + "o", width, heads * 128))


def _gokazen(case, w, tokens, wanted):
    c, width = config_of(case), case["width"]
    x = w("embed", VOCAB, width)[tokens]
    streams = [x, x.clone()]
    for i, layer in enumerate(c["layers"]):
        p = f"l{i}."
        for q in (1, 2):
            take = w(f"{p}hc{q}.in", 2)
            h = _rms(take[0] * streams[0] + take[1] * streams[1]) * (1.0 + w(f"{p}norm{q}", width))
            if q == 2:
                y = _linear(torch.relu(_linear(h, w(p + "mlp.up", 3 * width, width))) ** 2, w(p + "mlp.down", width, 3 * width))
            else:
                y = (_lightning if layer["type"] == "lightning" else _latent)(h, w, p + "mix.", layer["mixer"], width)
            y = y * w(f"{p}ls{q}", width)
            mix, give = w(f"{p}hc{q}.mix", 2, 2), w(f"{p}hc{q}.out", 2)
            streams = [mix[0, t] * streams[0] + mix[1, t] * streams[1] + give[t] * y for t in (0, 1)]
    return _linear(_rms(wanted(streams[0] + streams[1])) * (1.0 + w("final.norm", width)), w("head", VOCAB, width))


def _layer_norm(x, weight_, bias):
    centred = x - x.mean(-1, keepdim=True)
    return centred / torch.sqrt((centred * centred).mean(-1, keepdim=True) + 1e-6) * weight_ + bias


def _clamped(h, w, p, ff, width, limit):
    g = torch.clamp(_linear(h, w(p + "gate", ff, width)), max=limit)
    u = torch.clamp(_linear(h, w(p + "up", ff, width)), -limit, limit)
    return _linear(g * torch.sigmoid(1.702 * g) * (u + 1.0), w(p + "down", width, ff))


def _experts(h, w, p, mlp, width):
    flat, top = h.reshape(-1, width), mlp["router"]["top"]
    logits = _linear(flat, w(p + "router", mlp["router"]["experts"], width)) + w(p + "router.b", mlp["router"]["experts"])
    picked, chosen = torch.topk(logits, top, dim=-1)
    shares = torch.softmax(picked, -1)
    out = _clamped(flat, w, p + "shared.", mlp["shared"]["ff"], width, mlp["shared"]["limit"])
    for e in range(mlp["router"]["experts"]):
        rows, place = torch.nonzero(chosen == e, as_tuple=True)
        if len(rows):
            y = _clamped(flat[rows], w, f"{p}e{e}.", mlp["expert"]["ff"], width, mlp["expert"]["limit"])
            out.index_add_(0, rows, shares[rows, place][:, None] * y)
    return out.reshape(h.shape)


def _convolved_attention(h, w, p, m, width):
    kv = m["kv_heads"] * 128
    q, k, v = (_conv(_linear(h, w(p + s, n, width)), w(p + s + ".conv", n, m["conv"])) for s, n in (("q", width), ("k", kv), ("v", kv)))
    q, k = _rms(q) * w(p + "q.norm", width), _rms(k) * w(p + "k.norm", kv)
    angles = _angles(h.shape[1], m["rot"]["dims"], m["rot"]["base"])
    o = _attend(_turn(_heads(q, m["heads"]), angles, True), _turn(_heads(k, m["kv_heads"]), angles, True), _heads(v, m["kv_heads"]), m["scale"])
    return _linear(o * torch.sigmoid(_linear(h, w(p + "g", width, width))), w(p + "o", width, width))


def _mamba2(h, w, p, m, width):
    heads, groups, n = m["heads"], m["groups"], m["state"]
    inner, per = heads * m["vdim"], heads // groups
    both = inner + 2 * groups * n
    z, xbc, dt = _linear(h, w(p + "in", inner + both + heads, width)).split([inner, both, heads], -1)
    xbc = _silu(_conv(xbc, w(p + "conv", both, m["conv"])) + w(p + "conv.b", both))
    x = _heads(xbc[..., :inner], heads)
    b = _heads(xbc[..., inner:inner + groups * n], groups).repeat_interleave(per, 2)
    c = _heads(xbc[..., inner + groups * n:], groups).repeat_interleave(per, 2)
    dt = torch.nn.functional.softplus(dt + w(p + "dt_bias", heads))
    decay = torch.exp(-torch.exp(w(p + "A_log", heads)) * dt)
    state = torch.zeros(h.shape[0], heads, n, m["vdim"], dtype=torch.float64, device=DEVICE)
    y = torch.empty_like(x)
    for t in range(h.shape[1]):
        state = decay[:, t, :, None, None] * state + b[:, t, :, :, None] * (dt[:, t, :, None] * x[:, t])[:, :, None, :]
        y[:, t] = (c[:, t, :, None, :] @ state)[:, :, 0]
    y = (y + w(p + "D", heads)[:, None] * x).reshape(z.shape) * _silu(z)
    y = _rms(_heads(y, m["norm_groups"])).reshape(z.shape) * w(p + "norm", inner)
    return _linear(y, w(p + "o", width, inner))


def _pudorax(case, w, tokens, wanted):
    c, width = config_of(case), case["width"]
    side, loop = c["token_side"]["dim"], c["loop"]
    x = w("embed", VOCAB, width)[tokens]
    x0, table = x, w("side.embed", VOCAB, len(c["layers"]) * side)
    inside = list(range(loop["start"], loop["stop"]))
    order = list(range(loop["start"])) + inside * loop["times"] + list(range(loop["stop"], len(c["layers"])))
    starts = {loop["start"] + i * len(inside) for i in range(loop["times"])}
    for run_, i in enumerate(order):
        layer, p = c["layers"][i], f"l{i}."
        if run_ in starts:
            x = _linear(torch.cat([x, x0], -1), w("loop.in", width, 2 * width))
        h = _layer_norm(x, w(p + "norm1", width), w(p + "norm1.b", width))
        x = x + (_convolved_attention if layer["type"] == "attention" else _mamba2)(h, w, p + "mix.", layer["mixer"], width)
        x = x + _experts(_layer_norm(x, w(p + "norm2", width), w(p + "norm2.b", width)), w, p + "mlp.", layer["mlp"], width)
        gate = torch.nn.functional.gelu(_linear(x, w(p + "side.gate", side, width)), approximate="tanh")
        gate = gate * table[tokens][..., i * side:(i + 1) * side]
        x = x + _rms(_linear(gate, w(p + "side.proj", width, side))) * w(p + "side.norm", width)
    logits = _linear(_layer_norm(wanted(x), w("final.norm", width), w("final.norm.b", width)), w("head", VOCAB, width))
    return c["logit_softcap"] * torch.tanh(logits / c["logit_softcap"])


def _biased_attention(h, w, p, m, width, kept, index):
    heads, groups = m["heads"], m["kv_heads"]
    if "kv_from" in m:
        k, v = kept[m["kv_from"]]
    else:
        k, v = kept[index] = tuple(_heads(_linear(h, w(p + s, groups * 128, width)), groups) for s in "kv")
    at = torch.arange(h.shape[1], device=DEVICE, dtype=torch.float64)
    warm = 1.0 + m["q_temp"]["coef"] * torch.log(torch.floor((at + 1) / m["q_temp"]["every"]) + 1.0)
    q = _heads(_linear(h, w(p + "q", width, width)), heads) * warm[:, None, None]
    slopes = [2.0 ** (-8.0 * (head + 1) / heads) for head in range(heads)]
    return _linear(_attend(q, k, v, m["scale"], window=m["mask"]["size"], slopes=slopes), w(p + "o", width, width))


def _chunk_attention(h, w, p, m, width):
    angles = _angles(h.shape[1], m["rot"]["dims"], m["rot"]["base"], m["rot"]["scaling"]["factor"])
    q, k, v = (_heads(_linear(h, w(p + s, n * 128, width)), n) for s, n in (("q", m["heads"]), ("k", m["kv_heads"]), ("v", m["kv_heads"])))
    o = _attend(_turn(q, angles, True), _turn(k, angles, True), v, m["scale"], chunk=m["mask"]["size"], cap=m["softcap"])
    return _linear(o, w(p + "o", width, width))


def _delta_rule(h, w, p, m, width):
    heads, groups = m["heads"], m["kv_heads"]
    q, k, v = (_heads(_silu(_conv(_linear(h, w(p + s, n * 128, width)), w(p + s + ".conv", n * 128, m["conv"]))), n)
               for s, n in (("q", groups), ("k", groups), ("v", heads)))
    q, k = ((x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(heads // groups, 2) for x in (q, k))
    q = q * 128 ** -0.5
    beta = torch.sigmoid(_linear(h, w(p + "b", heads, width)))
    g = torch.exp(-torch.exp(w(p + "A_log", heads)) * torch.nn.functional.softplus(_linear(h, w(p + "a", heads, width)) + w(p + "dt_bias", heads)))
    state = torch.zeros(h.shape[0], heads, 128, 128, dtype=torch.float64, device=DEVICE)
    o = torch.empty_like(v)
    for t in range(h.shape[1]):
        state = g[:, t, :, None, None] * state
        u = beta[:, t, :, None] * (v[:, t] - (k[:, t, :, None, :] @ state)[:, :, 0])
        state = state + k[:, t, :, :, None] * u[:, :, None, :]
        o[:, t] = (q[:, t, :, None, :] @ state)[:, :, 0]
    o = (_rms(o) * w(p + "norm", 128)).reshape(h.shape) * _silu(_linear(h, w(p + "g", width, width)))
    return _linear(o, w(p + "o", width, width))


def _time_mixing(h, w, p, m, width):
    heads, rank = m["heads"], m["decay_rank"]
    before = torch.nn.functional.pad(h, (0, 0, 1, 0))[:, :-1]
    z = {s: h + (before - h) * w(f"{p}mu.{s}", width) for s in "rkvgw"}
    r, k, v = (_heads(_linear(z[s], w(p + s, width, width)), heads) for s in "rkv")
    low = torch.tanh(_linear(z["w"], w(p + "w1", rank, width)))
    decay = _heads(torch.exp(-torch.exp(_linear(low, w(p + "w2", width, rank)) + w(p + "w0", width))), heads)
    u = w(p + "u", heads, 64)
    state = torch.zeros(h.shape[0], heads, 64, 64, dtype=torch.float64, device=DEVICE)
    o = torch.empty_like(v)
    for t in range(h.shape[1]):
        written = k[:, t, :, :, None] * v[:, t, :, None, :]
        o[:, t] = (r[:, t, :, None, :] @ (state + u[:, :, None] * written))[:, :, 0]
        state = decay[:, t, :, :, None] * state + written
    o = _rms(o).reshape(h.shape) * w(p + "norm", width) * _silu(_linear(z["g"], w(p + "g", width, width)))
    return _linear(o, w(p + "o", width, width))


def _vitudra(case, w, tokens, wanted):
    c, width, kept = config_of(case), case["width"], {}
    x = w("embed", VOCAB, width)[tokens]
    for i, layer in enumerate(c["layers"]):
        p, m = f"l{i}.", layer["mixer"]
        h = _rms(x) * (1.0 + w(p + "norm1", width))
        if layer["type"] == "attention":
            y = _biased_attention(h, w, p + "mix.", m, width, kept, i)
        elif layer["type"] == "wkv":
            y = _time_mixing(h, w, p + "mix.", m, width)
        else:
            y = (m["left_scale"] * _chunk_attention(h, w, p + "mix.left.", m["left"], width)
                 + m["right_scale"] * _delta_rule(h, w, p + "mix.right.", m["right"], width))
        ff = 3 * width
        gated = _silu(_linear(h, w(p + "mlp.gate", ff, width))) * _linear(h, w(p + "mlp.up", ff, width))
        x = x + c["residual_mult"] * (y + _linear(gated, w(p + "mlp.down", width, ff)))
    return _linear(_rms(wanted(x)) * (1.0 + w("final.norm", width)), w("head", VOCAB, width))


def _logits(case, w, sequences, want):
    """Logits of the last `want` positions of each sequence, sequence after sequence."""
    longest = max(len(s) for s in sequences)
    tokens = torch.zeros(len(sequences), longest, dtype=torch.long)
    for row, sequence in enumerate(sequences):
        tokens[row, :len(sequence)] = torch.tensor(sequence)
    forward = {"Qwen3": _qwen3, "Gokazen": _gokazen, "Pudorax": _pudorax, "Vitudra": _vitudra}[case["arch"]]
    return forward(case, w, tokens.to(DEVICE), lambda x: torch.cat([x[b, len(s) - want:len(s)] for b, s in enumerate(sequences)]))


def exact(case, seed):
    w, sequences = _Weights(case, seed), _prompts(case, seed)
    if case["do"] == "prefill":
        return _logits(case, w, sequences, case["want"])
    if case["do"] == "decode":
        return _logits(case, w, [s + [token] for s, token in zip(sequences, _given(case, seed)[0])], 1)
    if case["temperature"] > 0.0:
        return None      # which tokens are drawn is the framework's own choice of random numbers
    logits, chosen = [], []
    for _ in range(case["new"]):
        logits.append(_logits(case, w, sequences, 1))
        chosen.append(logits[-1].argmax(-1))
        sequences = [s + [int(token)] for s, token in zip(sequences, chosen[-1])]
    return {"logits": torch.stack(logits, 1), "tokens": torch.stack(chosen, 1)}
