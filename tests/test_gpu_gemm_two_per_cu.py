"""gemm_wide on workgroups of four waves, two per compute unit (tiles of 128x128 and 128x96): the sizes where a tile, a stage count
or the persistent grid ends, both blocks, all output types, with and without a bias, against the checks of
test_gpu_gemm_random_shapes (CPU checker on sampled rows, the whole output against a float64 product, guard rows)."""
import pytest

import test_gpu_gemm_random_shapes as shapes

pytestmark = pytest.mark.gpu

# (M, N, K, block, output type, bias, scratch memory), the tile; more than 512 tiles: a workgroup walks on to a second one
CASES = [
    ((1100, 4000, 640, 64, "bf16", True, False), "128x96"),      # 9 x 42 tiles, the last row 76 rows, the last column 64; five stages
    ((1030, 4100, 384, 64, "f32", True, False), "128x96"),       # an odd number of stages; a last row of six rows, a last column of 68
    ((700, 6001, 128, 64, "f16", False, False), "128x96"),       # one stage; rows of C off 16-byte boundaries
    ((3000, 1500, 1280, 128, "bf16", False, False), "128x96"),   # 24 x 16 tiles
    ((2049, 2400, 512, 128, "f16", True, False), "128x96"),      # a last row of tiles of one row, 25 whole columns
    ((2900, 2944, 640, 128, "f32", True, False), "128x96"),      # 713 tiles, an odd number of stages
    ((2054, 4090, 256, 64, "bf16", True, False), "128x96"),      # 731 tiles
    ((1900, 4090, 384, 64, "bf16", False, False), "128x128"),    # 15 x 32 tiles
    ((1900, 4090, 384, 128, "f32", False, False), "128x128"),
    ((2116, 2900, 256, 64, "f32", True, False), "128x128"),
    ((100, 50257, 512, 128, "bf16", True, False), "128x128"),    # one row of tiles, 393 of them; odd rows
    ((2178, 4090, 640, 64, "bf16", True, False), "128x128"),     # 576 tiles
    ((1806, 5000, 256, 128, "f16", True, False), "128x128"),     # 600 tiles
    ((3046, 4090, 384, 64, "f32", False, False), "128x128"),     # 768 tiles, an odd number of stages
]


@pytest.mark.parametrize("case,tile", CASES, ids=lambda c: c if isinstance(c, str) else f"{c[0]}x{c[1]}x{c[2]}-b{c[3]}-{c[4]}{'-bias' if c[5] else ''}")
def test_shape(case, tile):
    from blockwise_int8_linear_amd import _lib
    M, N, K, block = case[:4]
    assert _lib.load().bi8_gemm_kernel_name(M, N, K, K, K, block, 0).decode() == "gemm_wide_" + tile
    shapes.test_random_shape(case)
