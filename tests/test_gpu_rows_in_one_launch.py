"""Three to sixteen rows quantized by the workgroups that multiply with them (bi8x_linear_rows): the output of the quantizer and the GEMM as
two calls, bit for bit, on both kernels, at the ends of their tiles and of the rule's range, with the blocks that take the quantizer's
IEEE division."""
import ctypes

import pytest
import torch

from test_gpu_few_rows_specials import KINDS, _inputs, _same_bits
from util import DTYPES, config_as, kernel_launches

pytestmark = pytest.mark.gpu

_vp, _ci, _i64 = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64
CODE = {"f32": 0, "bf16": 1, "f16": 2}


def _call(x, wq, sw, bias, out, dtype, block, ldx):
    from blockwise_int8_linear_amd import _lib
    f = _lib.load().bi8x_linear_rows
    f.restype, f.argtypes = _ci, [_vp, _ci, _vp, _vp, _vp, _ci, _vp, _i64, _i64, _i64, _i64, _i64, _i64, _ci, _vp]
    return f(x.data_ptr(), CODE[dtype], wq.data_ptr(), sw.data_ptr(), bias.data_ptr() if bias is not None else None, CODE[dtype], out.data_ptr(), *out.shape, wq.shape[1], ldx,
             wq.shape[1], out.shape[1], block, torch.cuda.current_stream().cuda_stream)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("block", [64, 128])
@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("M,K,N", [(3, 128, 5), (16, 512, 4096), (3, 2688, 1000), (16, 512, 5120), (7, 1152, 5433), (4, 2048, 32768), (16, 1024, 777), (3, 5376, 130), (4, 4096, 6001)])
def test_output(M, K, N, dtype, block, kind):
    import blockwise_int8_linear_amd as pkg
    x, w = (t.to("cuda:0") for t in _inputs(M, K, N, block, dtype, kind))
    fits = M * K <= (8 if dtype == "f32" else 16) * 1024
    with config_as(pkg, block, DTYPES[dtype]), torch.no_grad():
        wq, sw = pkg.quantize_block_rowwise(w)
        xq, sx = pkg.quantize_block_rowwise(x)
        rows = torch.zeros(M, K + 64, dtype=x.dtype, device=x.device)       # (rows farther apart than they are long)
        rows[:, :K] = x
        for bias in (None, torch.randn(N, generator=torch.Generator().manual_seed(N)).to(DTYPES[dtype]).to(x.device)):
            want = pkg.int8_matmul_block64_rowwise_dequantize(xq, wq.t(), sx, sw, bias)
            for given, ld in ((x, K), (rows, K + 64)):
                out = torch.full((M, N), 7.0, dtype=x.dtype, device=x.device)
                assert _call(given, wq, sw, bias, out, dtype, block, ld) == (0 if fits else 6)      # 6: left to the two launches
                assert _same_bits(out.cpu(), want.cpu()) if fits else (out == 7).all()


def test_calls_that_are_left_to_two_launches():
    x, w, s = (torch.ones(32, 8192, device="cuda:0").to(t) for t in (torch.bfloat16, torch.int8, torch.float32))
    out = torch.full((32, 32), 7.0, dtype=torch.bfloat16, device="cuda:0")
    for M, K, block in ((2, 512, 128), (17, 512, 128), (16, 1152, 128), (4, 512, 32), (4, 500, 64)):
        assert _call(x, w[:, :K], s, None, out[:M], "bf16", block, 8192) == 6
    assert _call(x[:, 1:], w[:, :512], s, None, out[:4], "bf16", 128, 8192) == 6 and _call(x, w[:, :512], s, None, out[:4], "bf16", 128, 8190) == 6
    assert (out == 7).all()


@pytest.mark.parametrize("M,K,N,block,dtype,launches", [(3, 128, 5, 128, "bf16", 1), (16, 1024, 4096, 64, "bf16", 1), (4, 4096, 11008, 128, "f16", 1), (8, 1024, 777, 64, "f32", 1),
                                                        (16, 1152, 777, 64, "bf16", 2), (9, 1024, 777, 64, "f32", 2), (17, 512, 777, 64, "bf16", 2)])
def test_launches_of_the_layer(M, K, N, block, dtype, launches):
    """a layer in evaluation takes the one launch where the rule has it"""
    import blockwise_int8_linear_amd as pkg
    with config_as(pkg, block, DTYPES[dtype]), torch.no_grad():
        layer = pkg.BlockInt8Linear(K, N, device="cuda:0", dtype=DTYPES[dtype]).eval()
        layer.prepare_for_eval()
        x = torch.randn(M, K, device="cuda:0").to(DTYPES[dtype])
        assert kernel_launches(lambda: layer(x)) == launches
