"""gemv_rows with the quantizer in front (bi8_linear_few_rows): activations with blocks of zeros, subnormal and huge maxima, NaNs and
infinities among ordinary ones, biases of every type, columns that are no multiple of a wave's four, K up to six runs in flight; the
output of the quantizer and the GEMM as two calls, bit for bit."""
import pytest
import torch

from util import DTYPES, config_as

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("block", [64, 128])
@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("M,K,N", [(1, 128, 3), (1, 4096, 1022), (2, 3072, 517), (1, 8448, 70), (2, 640, 64)])
def test_output(M, K, N, dtype, block):
    import blockwise_int8_linear_amd as pkg
    from blockwise_int8_linear_amd import _lib
    g = torch.Generator().manual_seed(M + K + N)
    w = torch.randn(N, K, generator=g).mul_(0.02).to(DTYPES[dtype]).to("cuda:0")
    plain = torch.randn(M, K, generator=g)
    special = plain.clone()
    special[0, :block] = 0.0
    special[-1, K - block:] = 1e-39
    special[0, K // 2] = 3e38
    for value in (None, float("nan"), float("inf")):
        x = special.clone()
        if value is not None:
            x[-1, K // 3] = value
        for given in (x, plain):
            xd = given.to(DTYPES[dtype]).to("cuda:0")
            with config_as(pkg, block, DTYPES[dtype]), torch.no_grad():
                wq, sw = pkg.quantize_block_rowwise(w)
                xq, sx = pkg.quantize_block_rowwise(xd)
                for bias in (None, torch.randn(N, generator=g).to(DTYPES[dtype]).to("cuda:0")):
                    want = pkg.int8_matmul_block64_rowwise_dequantize(xq, wq.t(), sx, sw, bias)
                    out = torch.empty(M, N, dtype=DTYPES[dtype], device="cuda:0")
                    code = {"f32": 0, "bf16": 1, "f16": 2}[dtype]
                    rc = _lib.load().bi8_linear_few_rows(xd.data_ptr(), code, wq.data_ptr(), sw.data_ptr(), bias.data_ptr() if bias is not None else None, code,
                                                         out.data_ptr(), M, N, K, K, K, N, block, torch.cuda.current_stream().cuda_stream)
                    if rc == 6:                    # (more activations than the LDS holds)
                        continue
                    assert rc == 0
                    assert torch.equal(out.cpu().nan_to_num(7.0), want.cpu().nan_to_num(7.0))
