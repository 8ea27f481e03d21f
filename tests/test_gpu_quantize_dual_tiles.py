"""The dual quantizer's two kinds of tiles, those inside the matrix and those at its ends, in one workgroup one after the other: one
round of half tiles to several of whole ones, rows of x on and off 16-byte boundaries, codes and scales written past the matrix as
zeros, and blocks with NaNs, infinities, zeros, subnormal and huge maxima; both directions bit for bit those of the CPU checker."""
import ctypes

import pytest
import torch

import oracle
from util import DTYPES

pytestmark = pytest.mark.gpu


class Task(ctypes.Structure):
    _fields_ = [(n, ctypes.c_void_p) for n in ("x", "q", "qT", "scales", "scalesT")] + [(n, ctypes.c_int64) for n in ("R", "C", "ldx", "ldq", "ldqt", "Rp", "Cp")]


def _up(n, to=128):
    return (n + to - 1) // to * to


@pytest.mark.parametrize("block", [32, 64, 128])
@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("R,C", [(128, 64), (5, 3), (260, 1032), (1000, 2304), (129, 70001), (4230, 4104), (3000, 5003), (2048, 8192),
                                 (130, 199), (131, 202), (132, 204), (97, 205), (33, 206), (40, 9), (7, 4),           # rows that end anywhere in 16 bytes
                                 (1, 4096), (70, 4104), (127, 40000), (11008, 40),                        # no tile inside the matrix
                                 (300, 32768), (8192, 1000), (8200, 1032), (2048, 4096)])                 # two whole tiles for each CU, and those at the ends
def test_codes_and_scales(R, C, dtype, block):
    from blockwise_int8_linear_amd import _lib
    run = _lib.load().bi8x_quantize_dual
    run.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p]
    g = torch.Generator().manual_seed(R + C)
    x = torch.randn(R, C, generator=g)
    for value in (float("nan"), float("inf"), 3e38, -float("inf")):
        for _ in range(1 + R * C // 200000):
            x[int(torch.randint(0, R, (1,), generator=g)), int(torch.randint(0, C, (1,), generator=g))] = value
    x[:, C // 2] = 0.0
    x[R // 2] = 0.0
    x[R // 3, : C // 2] = 1e-39
    x = x.to(DTYPES[dtype])
    xd = x.to("cuda:0")
    Rp, Cp = _up(R), _up(C)
    q, qt = (torch.full((r, c), 99, dtype=torch.int8, device="cuda:0") for r, c in ((R, Cp), (C, Rp)))
    s, st = (torch.full((b // block, n), -1.0, device="cuda:0") for b, n in ((Cp, R), (Rp, C)))
    task = Task(xd.data_ptr(), q.data_ptr(), qt.data_ptr(), s.data_ptr(), st.data_ptr(), R, C, C, Cp, Rp, Rp, Cp)
    assert run(ctypes.byref(task), 1, {"f32": 0, "bf16": 1, "f16": 2}[dtype], block, None, torch.cuda.current_stream().cuda_stream) == 0
    for codes, scales, source, n, padded in ((q, s, x, C, Cp), (qt, st, x.t().contiguous(), R, Rp)):
        want_q, want_s = oracle.quantize_block_rowwise(source, block)
        codes, scales = codes.cpu(), scales.cpu()
        assert torch.equal(codes[:, :n], want_q) and not codes[:, n:].any()
        blocks = want_s.size(0)
        assert torch.equal(scales[:blocks].view(torch.int32), want_s.view(torch.int32)) and not scales[blocks:].any()
