"""The embedding's rows at widths of whole and cut pieces, and of tokens that are not in the table."""

import pytest
import torch

from test_gpu_kernels import K      # noqa: F401  (the fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width", [4, 6, 1020, 1024, 1028, 4100, 5120])
def test_embedding_rows(K, dtype, width):
    table = torch.randn(50, width, generator=torch.Generator().manual_seed(width)).to(dtype).cuda()
    tokens = torch.tensor([3, 49, 0, -1, 50, 17, 17], dtype=torch.int32, device="cuda:0")      # ids outside the table read row 0
    source = torch.tensor([-1, -1, 1, -1, -1, 0, -1], dtype=torch.int32, device="cuda:0")
    fed = torch.tensor([8, 9], dtype=torch.int32, device="cuda:0")
    out = torch.full((7, width), float("nan"), device="cuda:0")
    K.embed(tokens, table, out)
    assert torch.equal(out, table.float()[[3, 49, 0, 0, 0, 17, 17]])
    K.embed(tokens, table, out, token_src=source, fed_tokens=fed)
    assert torch.equal(out, table.float()[[3, 49, 9, 0, 0, 8, 17]])
