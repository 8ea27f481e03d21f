"""quantize_rowwise on codes as large as the L2s together and larger: the same codes and scales as row by row."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", [8192, 8193, 8199])          # 32 MiB of codes, one row more, a ragged last tile
def test_codes_around_the_threshold(rows, dtype):
    import blockwise_int8_linear_amd as pkg
    g = torch.Generator(device="cuda").manual_seed(rows)
    x = torch.randn(rows, 4096, generator=g, device="cuda").to(dtype)
    q, s = pkg.quantize_block_rowwise(x, 64)
    for first in range(0, rows, 4000):                         # a row's codes depend on that row only
        part_q, part_s = pkg.quantize_block_rowwise(x[first:first + 4000], 64)
        assert torch.equal(q[first:first + 4000], part_q) and torch.equal(s[:, first:first + 4000], part_s)
