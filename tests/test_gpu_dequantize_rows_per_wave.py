"""dequantize_rows_vec on one, two and four rows and one to four runs per wave (chosen by the number of 1 KiB runs of output rows): both
sides of the lines, ragged last rows, columns and blocks, aligned and odd row lengths; same bits as the oracle."""
import pytest
import torch

import oracle
from util import DTYPES, config_as

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("out", list(DTYPES))
@pytest.mark.parametrize("M,K,B", [(6144, 256, 64), (6145, 248, 64), (6147, 512, 128), (3001, 2056, 32), (2051, 4104, 128), (24577, 255, 64), (9001, 2049, 128), (5003, 1028, 256), (17001, 128, 32), (33001, 256, 64),
                                   (1027, 5003, 32), (1003, 3003, 64), (3007, 2049, 128), (7, 20001, 32), (1701, 5003, 32), (1201, 5003, 64), (1701, 5003, 16), (4501, 2049, 32)])
def test_values(M, K, B, out):
    import blockwise_int8_linear_amd as pkg
    g = torch.Generator().manual_seed(M + K)
    q = torch.randint(-127, 128, (M, K), generator=g, dtype=torch.int32).to(torch.int8)
    s = torch.rand(-(-K // B), M, generator=g) * 3
    with config_as(pkg, None, DTYPES[out]):
        got = pkg.dequantize_block_rowwise(q.cuda(), s.cuda(), B).cpu()
    want = oracle.dequantize_block_rowwise(q, s, B, DTYPES[out])
    bits = torch.int32 if out == "f32" else torch.int16
    assert torch.equal(got.view(bits), want.view(bits))
