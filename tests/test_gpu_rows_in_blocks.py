"""Row-wise kernels that write blocks of 16 rows take 16 neighbouring rows to an XCD: every row has to be written, once, whatever the
number of rows.  The blocks against the same kernel's rows, bit for bit."""

import pytest
import torch

from test_gpu_kernels import K, dev      # noqa: F401  (K: the fixture)

pytestmark = pytest.mark.gpu


def blocked(K, rows, width):
    out = K.to_blocked(torch.full((rows, width), float("nan"), dtype=torch.bfloat16, device="cuda:0"))
    assert out.block_rows == 16
    return out


@pytest.mark.parametrize("width", [64, 1024])
@pytest.mark.parametrize("rows", [1, 64, 127, 128, 129, 300, 513])
def test_rows_and_blocks_agree(K, rows, width):
    g = torch.Generator().manual_seed(rows + width)
    x, y = torch.randn(rows, width, generator=g), torch.randn(rows, width, generator=g)
    gate, w, b = torch.randn(rows, width, generator=g).bfloat16(), torch.randn(width, generator=g), torch.randn(width, generator=g)
    both = torch.randn(rows, 2 * width, generator=g).bfloat16()
    held = lambda t: dev(t.clone())
    calls = {
        "rmsnorm": lambda out: K.rmsnorm(held(x), dev(w), 1e-6, out),
        "layernorm": lambda out: K.layernorm(held(x), dev(w), dev(b), 1e-6, out),
        "sum_layernorm": lambda out: K.sum_layernorm(held(x), held(y), 0.7, dev(w), dev(b), 1e-6, out),
        "add_rmsnorm": lambda out: K.add_rmsnorm(held(x), held(y), dev(w), 1e-6, out),
        "streams": lambda out: K.streams_update_rmsnorm(held(x).unsqueeze(1).repeat(1, 2, 1), held(y), None, None, None, None, dev(w), 1e-6, out),
        "gated_rmsnorm": lambda out: K.gated_rmsnorm(held(x), dev(gate), 0, dev(w), 1e-6, out),
        "gated_group_rmsnorm": lambda out: K.gated_group_rmsnorm(held(x), dev(gate), 0, dev(w), 1e-6, out, 4),
        "relu_squared": lambda out: K.relu_squared(dev(gate), out),
        "clamped_glu": lambda out: K.clamped_glu(dev(both), out, 1.5, 1.702),
        "cast_concat": lambda out: K.cast_concat(held(x[:, :width // 2].contiguous()), held(y[:, :width // 2].contiguous()), out),
        "gelu_tanh": lambda out: K.gelu_tanh(dev(gate), out),
        "gate_heads": lambda out: K.gate_heads(dev(gate), width // 4, dev(both), width // 2, out, 4, width // 4),
    }
    for name, call in calls.items():
        in_rows, in_blocks = torch.full((rows, width), float("nan"), dtype=torch.bfloat16, device="cuda:0"), blocked(K, rows, width)
        call(in_rows)
        call(in_blocks)
        got = K.from_blocked(in_blocks)
        assert bool(torch.isfinite(in_rows.float()).all()) and torch.equal(got, in_rows), name
