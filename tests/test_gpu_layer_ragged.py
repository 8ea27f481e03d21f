"""The layer's forward and backward on sizes that are no multiples of 128, where the quantizers write their codes padded with zeros and
X and W are quantized in one launch: bit for bit the composition of the single operators on the same tensors (which pad by copies),
for the float weight, for weight codes made ahead of the call, and in evaluation; and against the CPU checker."""
import pytest
import torch

from oracle import oracle_torch
from util import DTYPES, config_as

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# (rows, in, out, block, type of x and G, type of W): edges of the 128-row and 64- or 128-column tiles, 64 past a multiple of 128,
# odd counts, one row of tiles, fewer tiles of one matrix than of the other, mixed types (two launches), blocks that are not padded
CASES = [
    (1000, 768, 600, 64, "bf16", "bf16"), (129, 576, 1000, 64, "f32", "f32"), (127, 320, 641, 128, "f16", "f16"), (65, 192, 4097, 64, "bf16", "bf16"),
    (300, 1088, 257, 128, "f32", "f32"), (1000, 513, 777, 64, "bf16", "bf16"), (2050, 64, 129, 32, "f16", "f16"), (77, 640, 384, 128, "bf16", "f32"),
    (5, 448, 2000, 64, "bf16", "bf16"), (200, 1000, 300, 256, "f32", "f32"), (200, 384, 300, 48, "bf16", "bf16"),
]


@pytest.mark.parametrize("scale_type", [torch.float32, torch.bfloat16], ids=["scales_f32", "scales_bf16"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}x{c[1]}x{c[2]}-b{c[3]}-{c[4]}-{c[5]}")
def test_layer_is_the_composition_of_its_operators(case, scale_type):
    import blockwise_int8_linear_amd as pkg
    M, K, N, block, xt, wt = case
    g = torch.Generator().manual_seed(M + K + N)
    x = torch.randn(M, K, generator=g).to(DTYPES[xt]).to(DEV).requires_grad_(True)
    w = (torch.randn(N, K, generator=g) * 0.05).to(DTYPES[wt]).to(DEV).requires_grad_(True)
    b = torch.randn(N, generator=g).to(DTYPES[wt]).to(DEV).requires_grad_(True)
    G = torch.randn(M, N, generator=g).to(DTYPES[xt]).to(DEV)
    with config_as(pkg, block, DTYPES[xt]):
        cfg = pkg.block_linear_config
        cfg.SHARED_EXP_TORCH_TYPE = scale_type
        try:
            mul, q, qt = pkg.int8_matmul_block64_rowwise_dequantize, pkg.quantize_block_rowwise, pkg.quantize_block_transposed
            y = pkg.blockwise_int8_linear.apply(x, w, b)
            y.backward(G)
            with torch.no_grad():
                (xq, xs), (wq, ws), (gq, gs) = q(x), q(w), q(G)
                (xtq, xts), (wtq, wts), (gtq, gts) = qt(x), qt(w), qt(G)
                want = mul(xq, wq.t(), xs, ws, b), mul(gq, wtq.t(), gs, wts), mul(gtq, xtq.t(), gts, xts)
            assert xq.is_cuda and torch.equal(y, want[0]) and torch.equal(x.grad, want[1].to(x.dtype)) and torch.equal(w.grad, want[2].to(w.dtype))
            assert (b.grad.double() - G.double().sum(0)).abs().max() <= (2.0 ** -8 if xt != "f32" else 1e-5) * G.double().abs().sum(0).max()
            # only one of the gradients
            x2, w2 = x.detach().requires_grad_(True), w.detach().requires_grad_(True)
            pkg.blockwise_int8_linear.apply(x2, w.detach(), None).backward(G)
            pkg.blockwise_int8_linear.apply(x.detach(), w2, None).backward(G)
            assert torch.equal(x2.grad, x.grad) and torch.equal(w2.grad, w.grad)
            # weight codes made ahead: as the quantizers return them, and as views of padded rows
            for codes in ((wq, ws, wtq, wts), pkg.quantize_weight_for_training(w)[:4]):
                x3, w3 = x.detach().requires_grad_(True), w.detach().requires_grad_(True)
                y3 = pkg.blockwise_int8_linear_Wint8.apply(x3, codes[0], codes[1], b.detach(), codes[2], codes[3], w3)
                y3.backward(G)
                assert torch.equal(y3, y) and torch.equal(x3.grad, x.grad) and torch.equal(w3.grad, w.grad)
            # evaluation (three dimensions)
            lin = pkg.BlockInt8Linear(K, N, True, DEV, DTYPES[wt]).eval()
            with torch.no_grad():
                lin.weight.copy_(w)
                lin.bias.copy_(b)
                assert torch.equal(lin(x.detach().view(1, M, K)), y.view(1, M, N))
        finally:
            cfg.SHARED_EXP_TORCH_TYPE = torch.float32
        if scale_type == torch.float32:
            ref = oracle_torch.int8_matmul_block_dequantize(xq.cpu(), wq.cpu(), xs.cpu(), ws.cpu(), block, b.detach().cpu(), DTYPES[xt])
            unit = {"f32": 4e-6, "bf16": 1.6e-2, "f16": 2e-3}[xt]        # the product's and the sum's rounding at the largest magnitude
            assert (y.detach().cpu().double() - ref.double()).abs().max() <= unit * ref.double().abs().max()


# (rows, in, out): fewer than 2^22 multiplications in every product, contractions that are no multiples of 128
SMALL = [(70, 192, 130), (100, 64, 64), (500, 72, 100), (20, 320, 400), (5, 200, 300), (1, 192, 130)]


@pytest.mark.parametrize("block", [32, 64, 128])
@pytest.mark.parametrize("case", SMALL, ids=lambda c: "x".join(map(str, c)))
def test_small_products_take_the_scales_as_they_are(case, block):
    """An infinite column scale gives infinities, not a column of NaN, and the column scales are not rounded: fp32 results within three
    roundings of their products and sums (2-norm: 2^-24 each at most, rms less than half of that) plus one per K-block."""
    import blockwise_int8_linear_amd as pkg
    M, K, N = case
    g = torch.Generator().manual_seed(M + K + N)
    x = torch.randn(M, K, generator=g).to(DEV).requires_grad_(True)
    w = (torch.randn(N, K, generator=g) * 0.05).to(DEV).requires_grad_(True)
    G = torch.randn(M, N, generator=g).to(DEV)

    def exact(a, sa, b, sb):
        out = 0
        for j in range(sa.shape[0]):
            cols = slice(j * block, (j + 1) * block)
            out = out + (a[:, cols].double() @ b[:, cols].double().t()) * sa[j].double()[:, None] * sb[j].double()[None, :]
        return out / 127.0 ** 2

    with config_as(pkg, block, torch.float32):
        mul, q, qt = pkg.int8_matmul_block64_rowwise_dequantize, pkg.quantize_block_rowwise, pkg.quantize_block_transposed
        y = pkg.blockwise_int8_linear.apply(x, w, None)
        y.backward(G)
        with torch.no_grad():
            (xq, xs), (wq, ws), (gq, gs) = q(x), q(w), q(G)
            (xtq, xts), (wtq, wts), (gtq, gts) = qt(x), qt(w), qt(G)
            products = ((y.detach(), (xq, xs, wq, ws)), (x.grad, (gq, gs, wtq, wts)), (w.grad, (gtq, gts, xtq, xts)))
            for got, (a, sa, b, sb) in products:
                want = exact(a, sa, b, sb)
                assert (got.double() - want).norm() <= 0.5 * (3 + sa.shape[0]) * 2.0 ** -24 * want.norm()
                if a.shape[0] > 64:
                    assert torch.equal(got, mul(a, b.t(), sa, sb))
            ws = ws.clone()
            ws[-1, 2] = float("inf")
            ref = oracle_torch.int8_matmul_block_dequantize(xq.cpu(), wq.cpu(), xs.cpu(), ws.cpu(), block, None, torch.float32)
            assert ref[:, 2].isinf().any()
            got = pkg.blockwise_int8_linear_Wint8.apply(x.detach(), wq, ws, None, wtq, wts).cpu()
        assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got[ref.isinf()], ref[ref.isinf()])


@pytest.mark.parametrize("kept", [False, True], ids=["evaluation", "kept_codes"])
def test_scales_of_another_type_leave_the_weight_codes_where_they_are(kept):
    """the scales are converted for the call, the codes (the layer's memory) are not copied"""
    import blockwise_int8_linear_amd as pkg
    with config_as(pkg, 64, torch.bfloat16):
        cfg = pkg.block_linear_config
        cfg.SHARED_EXP_TORCH_TYPE = torch.bfloat16
        try:
            K, N = 2048, 4096
            lin = pkg.BlockInt8Linear(K, N, False, DEV, torch.bfloat16, quantized_weight_training=kept).train(kept)
            x = torch.randn(24, K, device=DEV, dtype=torch.bfloat16)
            with torch.no_grad():
                lin(x)
                torch.cuda.synchronize()
                torch.cuda.reset_peak_memory_stats()
                before = torch.cuda.memory_allocated()
                lin(x)
            assert torch.cuda.max_memory_allocated() - before < N * K // 2
        finally:
            cfg.SHARED_EXP_TORCH_TYPE = torch.float32
