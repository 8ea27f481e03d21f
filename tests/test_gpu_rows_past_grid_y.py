"""quantize_rows_vec and dequantize_rows_vec on more row tiles than one slice of the grid holds (32768): the last slice lies partly past
the matrix' rows.  Same bits as the oracle, nothing written behind the codes, scales and outputs."""
import pytest
import torch

import oracle
from util import DTYPES

pytestmark = pytest.mark.gpu
CODE = {"f32": 0, "bf16": 1, "f16": 2}
GUARD = 4096


def _guarded(n, dtype, value):
    return torch.full((n + GUARD,), value, dtype=dtype, device="cuda:0")


# rows per tile: 4 (one row per wave), 8 (two), 16 (four)
@pytest.mark.parametrize("M,K,dtype,block,rows", [(131077, 17, "bf16", 128, 4), (131075, 19, "f32", 32, 4), (262147, 17, "bf16", 32, 8), (524300, 64, "bf16", 32, 16),
                                                  (524301, 32, "f32", 32, 16)])
def test_quantize(M, K, dtype, block, rows):
    from blockwise_int8_linear_amd import _lib
    assert -(M // -rows) > 32768                   # (in more than one slice)
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(M)).to(DTYPES[dtype])
    nblk = -(K // -block)
    xd, q, s = x.to("cuda:0"), _guarded(M * K, torch.int8, 99), _guarded(nblk * M, torch.float32, -1.0)
    rc = _lib.load().bi8_quantize_rowwise(xd.data_ptr(), CODE[dtype], q.data_ptr(), s.data_ptr(), M, K, K, K, block, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    want_q, want_s = oracle.quantize_block_rowwise(x, block)
    q, s = q.cpu(), s.cpu()
    assert torch.equal(q[:M * K].view(M, K), want_q) and torch.equal(s[:nblk * M].view(nblk, M).view(torch.int32), want_s.view(torch.int32))
    assert (q[M * K:] == 99).all() and (s[nblk * M:] == -1.0).all()


@pytest.mark.parametrize("M,K,out,block,rows", [(524300, 64, "bf16", 32, 16), (524301, 64, "f32", 64, 16), (524300, 23, "f16", 8, 16), (262149, 256, "f32", 64, 8)])
def test_dequantize(M, K, out, block, rows):
    from blockwise_int8_linear_amd import _lib
    assert -(M // -rows) > 32768
    g = torch.Generator().manual_seed(M)
    q = torch.randint(-127, 128, (M, K), generator=g, dtype=torch.int8)
    s = torch.rand(-(K // -block), M, generator=g)
    qd, sd, o = q.to("cuda:0"), s.to("cuda:0"), _guarded(M * K, DTYPES[out], 99.0)
    rc = _lib.load().bi8_dequantize_rowwise(qd.data_ptr(), sd.data_ptr(), o.data_ptr(), CODE[out], M, K, K, K, block, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    o = o.cpu()
    bits = torch.int32 if out == "f32" else torch.int16
    assert torch.equal(o[:M * K].view(M, K).view(bits), oracle.dequantize_block_rowwise(q, s, block, DTYPES[out]).view(bits))
    assert (o[M * K:] == 99.0).all()
