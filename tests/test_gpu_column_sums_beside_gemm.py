"""The bias gradient of a layer, whose last step runs beside a GEMM of the backward pass (gemm_panel, gemm_wide_pair, splitk_reduce) or in a launch of its
own: the bits of bi8_quantize_dual_colsum, whichever kernel it is, at numbers of columns around those of a workgroup and of rows around a tile's 128."""
import ctypes

import pytest
import torch

from util import DTYPES, config_as, kernel_launches

pytestmark = pytest.mark.gpu

# tokens, in, out, block, the kernel of grad_W (the pair's: of both)
CASES = [
    (256, 1024, 1024, 64, "gemm_panel"), (129, 640, 767, 128, "gemm_panel"), (2300, 512, 769, 128, "gemm_panel"), (640, 768, 2304, 64, "gemm_panel"),
    (549, 1410, 642, 64, "pair"), (667, 5184, 1283, 64, "pair"), (776, 7103, 1280, 128, "pair"), (2374, 1472, 3009, 128, "pair"), (458, 2689, 896, 128, "pair"),
    (8192, 768, 3072, 64, "gemm_wide_256x128_splitk"), (6259, 832, 768, 128, "gemm_tile_128x128_splitk"), (6000, 2048, 100, 128, "gemm_panel_splitk"),
    (2048, 2048, 2049, 128, "pair"), (4495, 317, 342, 64, "gemm_tile_64x128_splitk"), (7677, 419, 8864, 128, "gemm_wide_256x192_splitk"),
    (147, 2736, 1644, 128, "gemm_wide_256x128"), (137, 2720, 7309, 128, "gemm_wide+gemm_wide_256x128"), (300, 300, 50, 64, None),
]


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("tokens,k,n,block,kernel", CASES)
def test_bits(tokens, k, n, block, kernel, dtype):
    import blockwise_int8_linear_amd as pkg
    from blockwise_int8_linear_amd import _lib, ops
    import test_gpu_gemm_pair as pairs
    lib, up = _lib.load(), lambda v: -(-v // 128) * 128
    pair = pairs._name(pairs.with_types(lib), pairs._sizes(tokens, k, n), block)
    if kernel == "pair":
        assert pair
    elif kernel:
        assert not pair and lib.bi8_gemm_kernel_name(n, k, up(tokens), up(tokens), up(tokens), block, lib.bi8_gemm_workspace_bytes(n, k, up(tokens), block)).decode() == kernel
    gen = torch.Generator(device="cuda:0").manual_seed(tokens + k + n)
    x, w, g = (torch.randn(*s, generator=gen, device="cuda:0").to(DTYPES[dtype]) for s in ((tokens, k), (n, k), (tokens, n)))
    bias = torch.zeros(n, dtype=DTYPES[dtype], device="cuda:0", requires_grad=True)
    x.requires_grad_(True)
    w.requires_grad_(True)
    with config_as(pkg, block, DTYPES[dtype]):
        pkg.blockwise_int8_linear.apply(x, w, bias).backward(g)
        want = ops.quantize_block_dual_colsum(g, block)[4]
        x.grad, w.grad, alone = None, None, bias.grad
        bias.grad = None
        pkg.blockwise_int8_linear.apply(x, w, bias).backward(g)
    assert torch.equal(alone, want) and torch.equal(bias.grad, want)


class _ColSums(ctypes.Structure):
    _fields_ = [("part", ctypes.c_void_p), ("out", ctypes.c_void_p), ("dtype", ctypes.c_int), ("R", ctypes.c_int64), ("C", ctypes.c_int64)]


@pytest.mark.parametrize("tokens,k,n,block,kernel", [c for c in CASES if c[4]])
def test_launches(tokens, k, n, block, kernel):
    """the sums take no launch of their own beside gemm_panel, the pair and a split's reduction, and one beside the other kernels"""
    from blockwise_int8_linear_amd import _lib
    import test_gpu_gemm_pair as pairs
    lib, dev = pairs.with_types(_lib.load()), "cuda:0"
    sizes = [(m, c, pairs._up(d, 128)) for m, c, d in pairs._sizes(tokens, k, n)]
    part, out = torch.zeros(-(-tokens // 128), n, device=dev), torch.empty(n, device=dev)
    sums = _ColSums(part.data_ptr(), out.data_ptr(), 0, tokens, n)
    held, problems = [], []
    for M, N, K in sizes:
        held.append([torch.zeros(M, K, dtype=torch.int8, device=dev), torch.zeros(N, K, dtype=torch.int8, device=dev), torch.ones(K // block, M, device=dev),
                     torch.ones(K // block, N, device=dev), torch.empty(M, N, dtype=torch.bfloat16, device=dev)])
        problems.append(pairs.Gemm(*(t.data_ptr() for t in held[-1]), M, N, K, K, K, K, N))
    if kernel == "pair":
        both = (pairs.Gemm * 2)(*problems)

        def call():
            assert lib.bi8x_gemm_pair(ctypes.byref(both), 1, block, ctypes.byref(sums), torch.cuda.current_stream().cuda_stream) == 0

        assert kernel_launches(call) == 1
        return
    M, N, K = sizes[1]
    need = lib.bi8_gemm_workspace_bytes(M, N, K, block)
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device=dev)
    lib.bi8x_gemm_sums.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_void_p, ctypes.c_int64, ctypes.c_void_p, ctypes.c_void_p]

    def call():
        assert lib.bi8x_gemm_sums(ctypes.byref(problems[1]), 1, block, ws.data_ptr() if need else None, need, ctypes.byref(sums), torch.cuda.current_stream().cuda_stream) == 0

    assert kernel_launches(call) == (1 if kernel == "gemm_panel" else 2)      # (a split: with its reduction; the others: with bi8x_colsum_finish)
