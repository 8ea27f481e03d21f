"""quantize_rowwise on one, two and four rows per wave (chosen by the number of 1 KiB runs of rows): ragged last rows and columns,
aligned and odd row lengths, all input types, with blocks of zeros, NaNs, infinities, subnormal and huge maxima among ordinary ones;
codes and scales bit for bit those of the CPU checker."""
import pytest
import torch

import oracle
from util import DTYPES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("block", [8, 32, 128, 256])
@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("M,K", [(1, 256), (7, 264), (1025, 1544), (1023, 4104), (2051, 4104), (5003, 2056), (1030, 5003), (3, 17), (4097, 128), (9301, 523), (3101, 3011), (18501, 203)])
def test_codes_and_scales(M, K, dtype, block):
    import blockwise_int8_linear_amd as pkg
    g = torch.Generator().manual_seed(M + K)
    x = torch.randn(M, K, generator=g)
    for value in (0.0, float("nan"), float("inf"), 1e-39, 3e38, -float("inf")):        # whole blocks, then single elements
        rows = torch.randint(0, M, (1 + M // 50,), generator=g)
        for r in rows.tolist():
            c = int(torch.randint(0, K, (1,), generator=g))
            if value == 0.0 or value == 1e-39:
                x[r, c // block * block:(c // block + 1) * block] = value
            else:
                x[r, c] = value
    x = x.to(DTYPES[dtype])
    q, s = pkg.quantize_block_rowwise(x.to("cuda:0"), block)
    qo, so = oracle.quantize_block_rowwise(x, block)
    assert torch.equal(q.cpu(), qo)
    assert torch.equal(s.cpu().view(torch.int32), so.view(torch.int32))
