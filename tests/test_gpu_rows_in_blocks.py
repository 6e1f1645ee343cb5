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


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,width", [(128, 4096), (129, 4128), (2049, 256), (2100, 264), (530, 1000), (530, 4096), (40, 16640), (16, 33280)])
def test_pieces_and_elements_agree(K, dtype, rows, width):
    """Element-wise kernels take a thread a piece of 16 bytes from a size on and a thread an element below it: the step's first rows
    alone are below it, so that both run the same rows; widths of fewer pieces than a workgroup's threads and of more, a last piece in
    the middle of one.  Bit for bit."""
    g = torch.Generator().manual_seed(rows + width)
    few = max(1, 400_000 // (8 * width))
    x, both = (torch.randn(rows, n, generator=g).to(dtype).cuda() for n in (width, 2 * width))
    f32 = torch.randn(rows, width, generator=g).cuda()
    calls = {
        "relu_squared": lambda n, out: K.relu_squared(x[:n], out),
        "gelu_tanh": lambda n, out: K.gelu_tanh(x[:n], out),
        "clamped_glu": lambda n, out: K.clamped_glu(both[:n], out, 1.5, 1.702),
        "cast_concat": lambda n, out: K.cast_concat(f32[:n], None, out),
        "gate_heads": lambda n, out: K.gate_heads(x[:n], width // 8, both[:n], width, out, 8, width // 8),
    }
    for name, call in calls.items():
        whole, part = (torch.full((n, width), float("nan"), dtype=dtype, device="cuda:0") for n in (rows, few))
        call(rows, whole)
        call(few, part)
        assert bool(torch.isfinite(whole.float()).all()) and torch.equal(whole[:few], part), name
        if dtype == torch.bfloat16 and width % 32 == 0:
            out = blocked(K, rows, width)
            call(rows, out)
            assert torch.equal(K.from_blocked(out), whole), name
