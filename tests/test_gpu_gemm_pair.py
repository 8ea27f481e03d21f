"""Two GEMMs in one launch (bi8x_gemm_pair): every tile that the rule chooses, both blocks, ragged edges, several tiles per workgroup, an odd number
of stages and rows of W that hold less than the padded contraction; the bits of the one-pass kernels, and nothing beside the outputs."""
import ctypes

import pytest
import torch

from util import DTYPES, config_as

_vp, _i64 = ctypes.c_void_p, ctypes.c_int64


class Gemm(ctypes.Structure):
    _fields_ = [(n, _vp) for n in ("A", "W", "sA", "sW", "C")] + [(n, _i64) for n in ("M", "N", "K", "kw", "lda", "ldw", "ldc")]


def with_types(lib):
    lib.bi8x_gemm_pair.argtypes = [_vp, ctypes.c_int, ctypes.c_int, _vp, _vp]
    lib.bi8x_gemm_pair_name.argtypes, lib.bi8x_gemm_pair_name.restype = [_vp, ctypes.c_int, ctypes.c_int], ctypes.c_char_p
    lib.bi8x_gemm.argtypes = [_vp] * 5 + [ctypes.c_int, _vp, ctypes.c_int] + [_i64] * 7 + [ctypes.c_int, _vp, _i64, _vp]
    return lib


@pytest.fixture(scope="module")
def lib():
    from blockwise_int8_linear_amd import _lib
    return with_types(_lib.load())


def _up(n, to):
    return -(-n // to) * to


def _sizes(tokens, k, n):
    """grad_X and grad_W of a layer as (M, N, contraction)"""
    return (tokens, k, n), (n, k, tokens)


def _name(lib, sizes, block, at=4096, dtype="bf16", **over):
    q = (Gemm * 2)(*(Gemm(at, at, at, at, at, m, n, _up(k, 128), _up(k, 128), _up(k, 128), _up(k, 128), n) for m, n, k in sizes))
    for field, value in over.items():
        setattr(q[1], field, value)
    return lib.bi8x_gemm_pair_name(ctypes.byref(q), ["f32", "bf16", "f16"].index(dtype), block).decode()


# tokens, in, out, block, the tile
CASES = [
    (418, 1731, 578, 64, "gemm_wide_128x96"),        # ragged rows and columns, rows of C off 16-byte boundaries
    (1497, 2001, 1500, 64, "gemm_wide_128x96"),      # more tiles than one round of either share
    (133, 9536, 573, 128, "gemm_wide_128x96"),       # a second problem of two stages
    (937, 1664, 897, 64, "gemm_wide_128x128"),
    (458, 2689, 896, 128, "gemm_wide_128x128"),
    (667, 5184, 1283, 64, "gemm_wide_256x128"),      # an odd number of stages
    (1328, 2304, 1664, 128, "gemm_wide_256x128"),
    (2136, 2368, 1746, 64, "gemm_wide_256x192"),
    (2374, 1472, 3009, 128, "gemm_wide_256x192"),
    (2420, 6656, 896, 64, "gemm_wide"),
    (776, 7103, 1280, 128, "gemm_wide"),             # several tiles per workgroup
]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("tokens,k,n,block,tile", CASES)
def test_bits_of_the_one_pass_kernels(lib, tokens, k, n, block, tile, dtype):
    sizes = _sizes(tokens, k, n)
    assert _name(lib, sizes, block) == tile
    gen = torch.Generator(device="cuda:0").manual_seed(tokens + k + n)
    stream, code = torch.cuda.current_stream().cuda_stream, ["f32", "bf16", "f16"].index(dtype)
    held, q, want, out = [], [], [], []
    for i, (M, N, K) in enumerate(sizes):
        kp, kw = _up(K, 128), _up(K, 16) if i == 0 else _up(K, 128)      # the first problem's W: a view of rows that are farther apart than kw
        A, W = (torch.randint(-127, 128, (rows, kp), dtype=torch.int8, generator=gen, device="cuda:0") for rows in (M, N))
        A[:, K:] = 0
        sa, sw = torch.rand(kp // block, M, generator=gen, device="cuda:0") + 0.01, torch.rand(-(-kw // block), N, generator=gen, device="cuda:0") + 0.01
        sa[-(-K // block):] = 0
        guard = torch.full((M + 2, N), 7.0, dtype=DTYPES[dtype], device="cuda:0")
        one = torch.empty(M, N, dtype=DTYPES[dtype], device="cuda:0")
        assert lib.bi8x_gemm(A.data_ptr(), W.data_ptr(), sa.data_ptr(), sw.data_ptr(), None, 0, one.data_ptr(), code, M, N, kp, kw, kp, kp, N, block, None, 0, stream) == 0
        held += [A, W, sa, sw]
        q.append(Gemm(A.data_ptr(), W.data_ptr(), sa.data_ptr(), sw.data_ptr(), guard[1:].data_ptr(), M, N, kp, kw, kp, kp, N))
        want.append(one)
        out.append(guard)
    pair = (Gemm * 2)(*q)
    for _ in range(2):
        assert lib.bi8x_gemm_pair(ctypes.byref(pair), code, block, None, stream) == 0
        for got, one in zip(out, want):
            assert torch.equal(got[1:-1], one) and (got[0] == 7).all() and (got[-1] == 7).all()
            got[1:-1] = 3.0


def test_where_the_rule_ends(lib):
    for tokens, k, n, block, _ in CASES:
        sizes = _sizes(tokens, k, n)
        assert _name(lib, sizes, 32) == _name(lib, sizes, 256) == ""
        for over in ({"A": 8}, {"sW": 2}, {"lda": _up(tokens, 128) + 8}, {"ldw": 1 << 23}, {"kw": 0}, {"kw": _up(tokens, 128) - 8}, {"K": _up(tokens, 128) - 64}, {"ldc": k - 1},
                     {"C": 0}, {"ldw": 16}, {"N": (1 << 31) - 1, "ldc": 1 << 31}):
            assert _name(lib, sizes, block, **over) == "", over
    # few rows in either problem, a contraction that wants its split, two gemm_panels, outputs that are little else than written
    for tokens, k, n, block in ((128, 9536, 573, 128), (937, 1664, 128, 64), (1141, 768, 19840, 64), (498, 896, 2304, 128), (4096, 4096, 11008, 128), (8192, 768, 3072, 64), (147, 10752, 13477, 64)):
        assert _name(lib, _sizes(tokens, k, n), block) == "", (tokens, k, n)
    # a gemm_panel of 60 stages or more, many outputs per stage beside a problem that fills the chip by itself (fp32 ones count twice), little to save at block 64
    for tokens, k, n, block, dtype in ((1016, 3456, 17984, 128, "bf16"), (1922, 1728, 14464, 128, "f16"), (1788, 2176, 21632, 128, "f32"), (695, 11328, 6144, 128, "bf16"),
                                       (796, 9472, 7708, 128, "f16"), (2021, 12096, 512, 128, "f32"), (6548, 10624, 1024, 64, "f32"), (292, 1472, 576, 64, "bf16")):
        assert _name(lib, _sizes(tokens, k, n), block, dtype=dtype) == "", (tokens, k, n)
    # ... and on the near side of these lines
    for tokens, k, n, block, dtype in ((7340, 3072, 832, 128, "f16"), (226, 11072, 1381, 128, "bf16"), (768, 8448, 3136, 128, "f32"), (323, 2304, 576, 64, "f16")):
        assert _name(lib, _sizes(tokens, k, n), block, dtype=dtype) != "", (tokens, k, n)


# layers of which one gradient by itself is summed in pieces of K (or has a rest that is)
PIECES = [
    (293, 5888, 8192, 64), (425, 4544, 8000, 128), (411, 5312, 5504, 128), (2584, 768, 4992, 128), (979, 2560, 5824, 128),      # 128x128 and 256x128 tiles
    (5676, 3008, 2496, 128), (5424, 4992, 3392, 64), (3314, 3264, 10303, 64),       # the rest of a cut
    (2091, 2240, 15296, 128), (8117, 896, 4800, 128),                               # 256x192 tiles
]


def _own(lib, sizes, block):
    return [lib.bi8_gemm_kernel_name(m, n, _up(k, 128), _up(k, 128), _up(k, 128), block, lib.bi8_gemm_workspace_bytes(m, n, _up(k, 128), block)).decode() for m, n, k in sizes]


def test_pieces_of_k_stay_pieces(lib):
    """one chain of sums over all of K has a larger error than its pieces: such a gradient keeps the launches it has by itself"""
    for tokens, k, n, block in PIECES:
        sizes = _sizes(tokens, k, n)
        assert any("splitk" in name for name in _own(lib, sizes, block)), (tokens, k, n)
        assert _name(lib, sizes, block) == "", (tokens, k, n)
    taken = 0
    for tokens in (129, 300, 511, 1000, 1500, 2600, 4100, 8000):
        for k in (512, 1111, 2304, 4992, 11008):
            for n in (640, 1999, 3456, 8320, 20000):
                for block in (64, 128):
                    sizes = _sizes(tokens, k, n)
                    if _name(lib, sizes, block):
                        taken += 1
                        assert not any("splitk" in name for name in _own(lib, sizes, block)), (tokens, k, n, block)
    assert taken > 50


@pytest.mark.gpu
@pytest.mark.parametrize("tokens,k,n,block", [c[:4] for c in CASES] + PIECES[:1] + PIECES[2:4] + PIECES[6:8] + PIECES[9:])
def test_bits_do_not_depend_on_the_other_gradient(tokens, k, n, block):
    """x and the weight differentiated together, and each alone"""
    import blockwise_int8_linear_amd as pkg
    gen = torch.Generator(device="cuda:0").manual_seed(tokens + k + n)
    x, w, g = (torch.randn(*s, generator=gen, device="cuda:0") for s in ((tokens, k), (n, k), (tokens, n)))
    got = {}
    with config_as(pkg, block, torch.float32):
        for which in ("xw", "x", "w"):
            leaves = {"x": x.clone().requires_grad_("x" in which), "w": w.clone().requires_grad_("w" in which)}
            pkg.blockwise_int8_linear.apply(leaves["x"], leaves["w"], None).backward(g)
            got[which] = {name: t.grad for name, t in leaves.items()}
    assert torch.equal(got["xw"]["x"], got["x"]["x"]) and torch.equal(got["xw"]["w"], got["w"]["w"])
