"""gemm_wide on tiles of 256x192 (one round of at most 256 of them, where 256x256 tiles would leave many CUs idle): ragged last rows and
columns of tiles, odd and even numbers of stages, both blocks, all output types, with and without a bias, rows of C off 16-byte
boundaries, against the checks of test_gpu_gemm_random_shapes (CPU checker on sampled rows, the whole output against a float64
product, guard rows)."""
import pytest

import test_gpu_gemm_random_shapes as shapes

pytestmark = pytest.mark.gpu

CASES = [
    (2944, 2944, 2048, 128, "bf16", False, False),     # 12 x 16 tiles, the last column of tiles 64 columns
    (2820, 3393, 1920, 128, "f16", True, False),       # a last row of tiles of four rows, rows of C of odd length, an odd number of stages
    (772, 10304, 1408, 128, "f32", True, False),       # 4 x 54 tiles
    (2007, 5697, 1920, 64, "bf16", True, False),       # 240 tiles
    (3071, 3900, 1152, 64, "f32", False, False),       # 252 tiles, a last column of tiles of 60 columns
    (1100, 9013, 2304, 64, "f16", False, False),       # 235 tiles, the last row of tiles 76 rows
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}x{c[1]}x{c[2]}-b{c[3]}-{c[4]}{'-bias' if c[5] else ''}")
def test_shape(case):
    from blockwise_int8_linear_amd import _lib
    M, N, K, block = case[:4]
    assert _lib.load().bi8_gemm_kernel_name(M, N, K, K, K, block, 0).decode() == "gemm_wide_256x192"
    shapes.test_random_shape(case)
