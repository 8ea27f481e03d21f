"""256x256 tiles and the 256x128 tiles of the rest in one launch (gemm_wide_rest): cut by rows and by columns, a lead of fewer tiles than workgroups and of
several rounds, ragged ends, odd numbers of stages, a single stage in all, with and without a bias, against the checks of
test_gpu_gemm_random_shapes (CPU checker on sampled rows, the whole output against a float64 product, guard rows)."""
import pytest
import torch

import test_gpu_gemm_random_shapes as shapes
from util import DTYPES, kernel_launches

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


# cuts whose rest is on other tiles: a launch of its own, or two where it is split over K
OTHER_CUTS = [(1300, 11008, 128, 64, "bf16", False, False, 2), (4128, 5000, 128, 64, "f32", True, False, 2), (2100, 8192, 4096, 128, "bf16", True, True, 3)]


@pytest.mark.parametrize("case", [c + (1,) for c in CASES] + OTHER_CUTS, ids=lambda c: f"{c[0]}x{c[1]}x{c[2]}-b{c[3]}-{c[7]}")
def test_launches(case):
    from blockwise_int8_linear_amd import _lib
    lib = _lib.load()
    M, N, K, block, dtype, with_bias, with_scratch, launches = case
    need = lib.bi8_gemm_workspace_bytes(M, N, K, block) if with_scratch else 0
    name = lib.bi8_gemm_kernel_name(M, N, K, K, K, block, need).decode()
    assert name.startswith("gemm_wide+") and (name == "gemm_wide+gemm_wide_256x128") == (launches == 1) and ("splitk" in name) == (launches == 3)
    dev = "cuda:0"
    A, W = (torch.zeros(rows, K, dtype=torch.int8, device=dev) for rows in (M, N))
    sa, sw = (torch.ones(K // block, rows, device=dev) for rows in (M, N))
    C, bias, ws = torch.empty(M, N, dtype=DTYPES[dtype], device=dev), torch.zeros(N, device=dev), torch.empty(max(need, 16), dtype=torch.uint8, device=dev)

    def call():
        assert lib.bi8_gemm_nt_dequant_ws(A.data_ptr(), W.data_ptr(), sa.data_ptr(), sw.data_ptr(), bias.data_ptr() if with_bias else None, 0, C.data_ptr(),
                                          list(DTYPES).index(dtype), M, N, K, K, K, N, block, ws.data_ptr() if need else None, need, torch.cuda.current_stream().cuda_stream) == 0

    assert kernel_launches(call) == launches
