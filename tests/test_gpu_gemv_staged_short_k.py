"""gemv_staged on contractions that end inside a turn of its ring of stages (one 128-byte chunk of K to a few per wave, workgroups of
four and of eight waves, one to four groups of rows), with and without a bias, against the checks of test_gpu_gemm_random_shapes."""
import pytest

import test_gpu_gemm_random_shapes as shapes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N", [(3, 100), (16, 4096), (17, 1000), (32, 4609), (16, 70001), (40, 2000)])
@pytest.mark.parametrize("K,block,out,bias", [(128, 64, "bf16", True), (384, 128, "f32", False), (1152, 64, "f16", True), (1280, 128, "bf16", False), (2176, 128, "f32", True)])
def test_shape(M, N, K, block, out, bias):
    from blockwise_int8_linear_amd import _lib
    if M > 32 and K < 1152:
        pytest.skip("gemm_panel's")
    assert _lib.load().bi8_gemm_kernel_name(M, N, K, K, K, block, 0).decode() == "gemv_staged"
    shapes.test_random_shape((M, N, K, block, out, bias, False))
