"""256x256 tiles and the 256x128 tiles of the rest in one launch (gemm_wide_rest): cut by rows and by columns, a lead of fewer tiles than workgroups and of
several rounds, ragged ends, odd numbers of stages, a single stage in all, with and without a bias, against the checks of
test_gpu_gemm_random_shapes (CPU checker on sampled rows, the whole output against a float64 product, guard rows)."""
import pytest

import test_gpu_gemm_random_shapes as shapes

pytestmark = pytest.mark.gpu

# (M, N, K, block, output type, bias, scratch memory)
CASES = [
    (4128, 5000, 512, 64, "bf16", True, False),      # a lead of 240 tiles: sixteen workgroups have none, and begin with the rest
    (5357, 4005, 768, 64, "f32", True, False),       # rows of C off 16-byte boundaries
    (4083, 5288, 640, 64, "f16", False, False),      # five stages
    (1547, 12056, 1024, 64, "f32", False, False),    # cut by columns
    (1300, 13733, 1024, 128, "bf16", True, False),
    (3727, 5858, 1024, 128, "f32", True, False),
    (2454, 8335, 512, 128, "f16", True, False),
    (11343, 4864, 256, 128, "bf16", False, False),   # three rounds of the lead, two stages
    (11343, 4864, 128, 128, "bf16", True, False),    # one stage
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}x{c[1]}x{c[2]}-b{c[3]}-{c[4]}{'-bias' if c[5] else ''}")
def test_shape(case):
    from blockwise_int8_linear_amd import _lib
    M, N, K, block = case[:4]
    assert _lib.load().bi8_gemm_kernel_name(M, N, K, K, K, block, 0).decode() == "gemm_wide+gemm_wide_256x128"
    shapes.test_random_shape(case)
