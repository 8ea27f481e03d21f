"""256x192 tiles on two pieces of K each: ragged edges, an odd number of stages, pieces of unequal length, the least tiles and K of the rule;
against the CPU checker on sampled rows and the one-pass kernel everywhere, and without the scratch memory or with the static array's."""
import pytest
import torch

from oracle import oracle_torch
from test_gpu_gemm_split import DEV, _problem, _run, lib  # noqa: F401
from util import DTYPES

pytestmark = pytest.mark.gpu

NAME = "gemm_wide_256x192_splitk"


@pytest.mark.parametrize("M,N,K,block,out", [(2305, 2049, 7168, 128, "f32"), (513, 8000, 7296, 128, "bf16"), (5600, 767, 14464, 64, "f16"), (1100, 4800, 14336, 64, "f32")])
def test_two_pieces(lib, M, N, K, block, out):  # noqa: F811
    A, W, sa, sw, bias = _problem(M, N, K, block, seed=M + N + K)
    want = lib.bi8_gemm_workspace_bytes(M, N, K, block)
    assert want == -(-M // 256) * -(-N // 192) * 2 * 256 * 192 * 4 and lib.bi8_gemm_kernel_name(M, N, K, K, K, block, want).decode() == NAME
    d = [t.to(DEV) for t in (A, W, sa, sw)]
    split, one = (_run(lib, *d, bias, block, out, ws) for ws in (want, want - 4))
    rows = torch.unique(torch.cat([torch.arange(0, M, M // 40), torch.tensor([M - 1])]))
    ref = oracle_torch.int8_matmul_block_dequantize(A[rows], W, sa[:, rows].contiguous(), sw, block, bias, torch.float32).double()
    P = oracle_torch.gemm_nt_partials(A[rows], W, block)
    mag = torch.zeros(len(rows), N, dtype=torch.float64)
    for j in range(K // block):
        mag += P[j].abs().double() * sa[j, rows].double()[:, None] * sw[j].double()[None, :]
    mag /= 127.0 * 127.0
    # per term 2^-22 for the column scale's rounding and 2^-24 for each of its sums and products (4e-6 of the terms' magnitudes holds them all with
    # the checker's own), then the output type's rounding, twice with a bias
    bound = (1e-5 if out == "f32" else 2.0 ** -7 if out == "bf16" else 2.0 ** -10) * (ref.abs() + bias.double().abs()[None, :]) + 4e-6 * mag + 1e-30
    assert ((split[rows.to(DEV)].cpu().double() - ref).abs() <= bound).all()
    if out == "f32":                               # sums of the same terms in another order
        assert (split - one).abs().max().item() <= 2e-5 * one.abs().max().item()
    assert torch.equal(split, _run(lib, *d, bias, block, out, want))
    static = torch.empty(M, N, dtype=DTYPES[out], device=DEV)
    b = bias.to(DEV)
    assert lib.bi8_gemm_nt_dequant_static(*(t.data_ptr() for t in d), b.data_ptr(), 0, static.data_ptr(), ["f32", "bf16", "f16"].index(out), M, N, K, K, K, N, block,
                                          torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(static, one)                # (planned with 32 MiB: one pass, as without scratch memory)


def test_where_the_rule_ends(lib):  # noqa: F811
    name = lambda *a: lib.bi8_gemm_kernel_name(a[0], a[1], a[2], a[2], a[2], a[3], a[4] if len(a) > 4 else 1 << 30).decode()  # noqa: E731
    assert name(8192, 768, 50304, 64) == NAME and name(2304, 2304, 7168, 128) == NAME
    for other in ((8192, 768, 7040, 128), (8192, 768, 14208, 64), (512, 11008, 32768, 128), (8192, 769, 16384, 128), (8192, 768, 16384, 32), (8192, 768, 16384, 128, 32 << 20)):
        assert name(*other) != NAME, other
    # at block 128 more than 110 tiles want a stage more each, except for up to 640 rows
    assert all(name(*taken) == NAME for taken in ((7814, 640, 9472, 128), (5440, 896, 7168, 128), (513, 8000, 7296, 128), (640, 8000, 7168, 128), (7832, 640, 14336, 64)))
    assert all(name(*other) != NAME for other in ((7832, 640, 8064, 128), (8128, 768, 8064, 128), (2560, 2240, 7168, 128), (641, 8000, 7168, 128)))
