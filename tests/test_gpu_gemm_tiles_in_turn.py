"""gemm_wide's workgroups on several tiles one after the other: a tile's outputs leave through LDS in front of loads and waits of the
next tile's, whole tiles by another path than tiles at the matrix' ends.  All four tiles, one stage of K to six, all output types, with
and without a bias, rows of C on and off 16-byte boundaries, against the checks of test_gpu_gemm_random_shapes (CPU checker on
sampled rows, the whole output against a float64 product, guard rows)."""
import pytest

import test_gpu_gemm_random_shapes as shapes

pytestmark = pytest.mark.gpu

# (M, N, K, block, output type, bias, scratch memory), the kernel; tiles per workgroup: two, or four of the last two
CASES = [
    ((3902, 6712, 384, 128, "bf16", False, False), "gemm_wide"),            # 432 tiles of 256x256, three stages, a last column of 56
    ((4613, 5824, 512, 128, "f32", True, False), "gemm_wide"),              # a last row of tiles of five rows
    ((3789, 6600, 640, 64, "f16", True, False), "gemm_wide"),
    ((5565, 4816, 768, 64, "bf16", True, False), "gemm_wide"),
    ((3601, 6136, 256, 128, "f32", False, False), "gemm_wide_256x128"),     # a last row of one row; two stages: the first pair is the last
    ((3666, 6241, 512, 64, "bf16", True, False), "gemm_wide_256x128"),      # rows of odd length
    ((3287, 4981, 768, 128, "f16", False, False), "gemm_wide_256x128"),
    ((4700, 4900, 128, 64, "f32", True, False), "gemm_wide_128x96"),        # one stage
    ((4700, 4901, 128, 128, "bf16", True, False), "gemm_wide_128x128"),
]


@pytest.mark.parametrize("case,kernel", CASES, ids=lambda c: c if isinstance(c, str) else f"{c[0]}x{c[1]}x{c[2]}-b{c[3]}-{c[4]}{'-bias' if c[5] else ''}")
def test_shape(case, kernel):
    from blockwise_int8_linear_amd import _lib
    M, N, K, block = case[:4]
    assert _lib.load().bi8_gemm_kernel_name(M, N, K, K, K, block, 0).decode() == kernel
    shapes.test_random_shape(case)
