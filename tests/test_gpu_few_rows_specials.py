"""gemv_rows with the quantizer in front (bi8_linear_few_rows): one kind of unusual block per case, of a size that leaves the outputs
finite (but for infinities), so that a wrong code or scale shows; biases of every type, columns that are no multiple of a wave's four, K up
to six runs in flight; the output of the quantizer and the GEMM as two calls, bit for bit."""
import pytest
import torch

from util import DTYPES, config_as

pytestmark = pytest.mark.gpu

SHAPES = [(1, 128, 3), (1, 4096, 1022), (2, 3072, 517), (1, 8448, 70), (2, 640, 64)]
KINDS = ["ordinary", "nan", "zero block", "subnormal", "huge", "inf"]
# factors of the activations and of W.  Maxima below 2^-60 or above 2^100 take the quantizer's IEEE division; fp16 has neither, and goes to
# the ends of its own range.
SUBNORMAL = {"f32": (1e-39, 1e4), "bf16": (1e-39, 1e4), "f16": (1e-6, 1e2)}
HUGE = {"f32": (2.0**101, 1e-20), "bf16": (2.0**101, 1e-20), "f16": (1e4, 1e-4)}


def _inputs(M, K, N, block, dtype, kind):
    """x [M,K], whose last row holds what `kind` says, and W [N,K], on the CPU"""
    g = torch.Generator().manual_seed(M + K + N)
    x, w = torch.randn(M, K, generator=g), torch.randn(N, K, generator=g)
    scale_w = 0.02
    row = x[-1]
    if kind == "nan":
        for at in (0, K // 3, K // 2, K - 1):
            row[at] = float("nan")
    elif kind == "zero block":
        row[:block] = 0.0
        row[K // 2 // block * block:][:block] = -0.0
        if K > 2 * block:
            row[K - block:] = 0.0
        row[K // 2] = 1.0                          # (a row of one block or two is not all zeros)
    elif kind in ("subnormal", "huge"):
        scale_x, scale_w = (SUBNORMAL if kind == "subnormal" else HUGE)[dtype]
        row.clamp_(-3.0, 3.0).mul_(scale_x)
    elif kind == "inf":
        row[K // 3] = float("inf")
        row[K - 1] = -float("inf")
    return x.to(DTYPES[dtype]), w.mul_(scale_w).to(DTYPES[dtype])


def _same_bits(a, b):
    bits = torch.int32 if a.dtype is torch.float32 else torch.int16
    return torch.equal(a.isnan(), b.isnan()) and torch.equal(a.view(bits)[~a.isnan()], b.view(bits)[~b.isnan()])


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("block", [64, 128])
@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("M,K,N", SHAPES)
def test_output(M, K, N, dtype, block, kind):
    import blockwise_int8_linear_amd as pkg
    from blockwise_int8_linear_amd import _lib
    from blockwise_int8_linear_amd.ops import _FEW_ROWS_LDS, _few_rows_lds
    x, w = (t.to("cuda:0") for t in _inputs(M, K, N, block, dtype, kind))
    code = {"f32": 0, "bf16": 1, "f16": 2}
    fits = _few_rows_lds(M, K, block, x.element_size()) <= _FEW_ROWS_LDS
    with config_as(pkg, block, DTYPES[dtype]), torch.no_grad():
        wq, sw = pkg.quantize_block_rowwise(w)
        xq, sx = pkg.quantize_block_rowwise(x)
        # (biases of every type, as large as the outputs of that row)
        size = float(pkg.int8_matmul_block64_rowwise_dequantize(xq, wq.t(), sx, sw, None)[0].float().abs().max())
        size = 1.0 if size != size or size == float("inf") else size
        for bias_type in (None, dtype, "f32"):
            bias = torch.randn(N, generator=torch.Generator().manual_seed(N)).mul_(size).to(DTYPES[bias_type]).to("cuda:0") if bias_type else None
            want = pkg.int8_matmul_block64_rowwise_dequantize(xq, wq.t(), sx, sw, bias)
            out = torch.empty(M, N, dtype=DTYPES[dtype], device="cuda:0")
            rc = _lib.load().bi8_linear_few_rows(x.data_ptr(), code[dtype], wq.data_ptr(), sw.data_ptr(), bias.data_ptr() if bias is not None else None,
                                                 code[bias_type or dtype], out.data_ptr(), M, N, K, K, K, N, block, torch.cuda.current_stream().cuda_stream)
            assert rc == (0 if fits else 6)        # 6: more activations than the LDS holds
            if fits:
                finite = want.isfinite()
                assert finite[:-1].all() and (not finite[-1].any() if kind == "inf" else finite[-1].all())
                assert want[finite].any() or kind == "inf"
                assert _same_bits(out.cpu(), want.cpu())
