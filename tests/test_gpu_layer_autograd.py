"""The layer in autograd beyond a plain backward pass: saved-tensor hooks, an output that no gradient reaches, traces, and the
transforms that it refuses."""
import pytest
import torch
import torch.autograd.forward_ad as fwad
import torch.utils.checkpoint

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(params=[False, True], ids=["float_weight", "kept_codes"])
def layer(request):
    import blockwise_int8_linear_amd as pkg
    block, pkg.block_linear_config.GROUP_SIZE = pkg.block_linear_config.GROUP_SIZE, 64
    dtype, pkg.block_linear_config.INPUT_OUTPUT_TORCH_TYPE = pkg.block_linear_config.INPUT_OUTPUT_TORCH_TYPE, torch.float32
    torch.manual_seed(0)
    yield pkg.BlockInt8Linear(192, 130, True, DEV, torch.float32, quantized_weight_training=request.param)
    pkg.block_linear_config.GROUP_SIZE, pkg.block_linear_config.INPUT_OUTPUT_TORCH_TYPE = block, dtype


def _grads(layer, x, g, call=None):
    x = x.detach().requires_grad_(True)
    layer.zero_grad(set_to_none=True)
    y = (call or layer)(x)
    y.backward(g)
    return [y.detach(), x.grad, layer.weight.grad, layer.bias.grad]


def test_saved_tensor_hooks_and_checkpointing(layer):
    x, g = torch.randn(70, 192, device=DEV), torch.randn(70, 130, device=DEV)
    want, seen = _grads(layer, x, g), []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append(t.shape) or t.cpu(), lambda t: t.to(DEV)):
        got = _grads(layer, x, g)
    assert seen and all(map(torch.equal, got, want))
    got = _grads(layer, x, g, lambda x: torch.utils.checkpoint.checkpoint(layer, x, use_reentrant=False))
    assert all(map(torch.equal, got, want))


def test_an_output_that_no_gradient_reaches(layer):
    class Stop(torch.autograd.Function):
        @staticmethod
        def forward(ctx, y):
            return y.clone()

        @staticmethod
        def backward(ctx, g):
            return None
    grads = _grads(layer, torch.randn(5, 192, device=DEV), torch.randn(5, 130, device=DEV), lambda x: Stop.apply(layer(x)))[1:]
    assert all(t is not None and not t.any() for t in grads)


def test_bias_gradient_is_differentiable_where_torch_computes_it(layer):
    g = torch.randn(5, 130, device=DEV, requires_grad=True)
    y = layer(torch.randn(5, 192, device=DEV))
    (gb,) = torch.autograd.grad(y, layer.bias, g, create_graph=True)
    gb.sum().backward()
    assert torch.equal(g.grad, torch.ones_like(g))


def test_a_trace_records_the_call(layer):
    x, other = torch.randn(7, 192, device=DEV), torch.randn(7, 192, device=DEV)
    if layer.quantized_weight_training:
        layer.prepare_for_quantized_weight_training()
    traced = torch.jit.trace(layer, x, check_trace=False)
    assert torch.equal(traced(other), layer(other))


@pytest.mark.parametrize("frozen", ["", "x", "weight", "weight bias", "x weight"])
def test_compiled_autograd(layer, frozen):
    from torch._dynamo import compiled_autograd
    enable = getattr(compiled_autograd, "_enable", None) or compiled_autograd.enable
    x, g = torch.randn(70, 192, device=DEV, requires_grad="x" not in frozen), torch.randn(70, 130, device=DEV)
    layer.weight.requires_grad_("weight" not in frozen)
    layer.bias.requires_grad_("bias" not in frozen)

    def grads(times=1):
        x.grad = None
        layer.zero_grad(set_to_none=True)
        y = layer(x)
        for i in range(times):
            y.backward(g, retain_graph=i + 1 < times)
        with pytest.raises(RuntimeError, match="second time"):
            y.backward(g)
        return [t.grad for t in (x, layer.weight, layer.bias) if t.requires_grad]
    want, twice = grads(), grads(2)
    for _ in range(2):
        with enable(torch.compile(backend="eager")):
            assert all(map(torch.equal, grads(), want)) and all(map(torch.equal, grads(2), twice))


def test_compiled_autograd_of_an_output_that_no_gradient_reaches(layer):
    from torch._dynamo import compiled_autograd
    enable = getattr(compiled_autograd, "_enable", None) or compiled_autograd.enable

    class Stop(torch.autograd.Function):
        @staticmethod
        def forward(ctx, y):
            return y.clone()

        @staticmethod
        def backward(ctx, g):
            return None
    x = torch.randn(5, 192, device=DEV, requires_grad=True)
    y = Stop.apply(layer(x))
    with enable(torch.compile(backend="eager")):
        y.backward(torch.randn(5, 130, device=DEV))
    assert all(t.grad is not None and not t.grad.any() for t in (x, layer.weight, layer.bias))


@pytest.mark.parametrize("traced", [False, True], ids=["eager", "traced"])
def test_a_graph_is_retained_where_that_is_asked_for(layer, traced):
    x, g = torch.randn(70, 192, device=DEV, requires_grad=True), torch.randn(70, 130, device=DEV)
    if layer.quantized_weight_training:
        layer.prepare_for_quantized_weight_training()
    seen = []

    class Keeps(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.layer = layer

        def forward(self, x):
            seen.append(self.layer(x))
            return seen[0]
    if traced:
        torch.jit.trace(Keeps(), x, check_trace=False)
    else:
        Keeps()(x)
    inputs = (x, layer.weight, layer.bias)
    first = torch.autograd.grad(seen[0], inputs, g, retain_graph=True)
    second = torch.autograd.grad(seen[0], inputs, g)
    assert all(map(torch.equal, first, second)) and torch.equal(first[0], _grads(layer, x, g)[1])
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(seen[0], inputs, g)


def test_refused_transforms(layer):
    x = torch.randn(3, 7, 192, device=DEV)
    with pytest.raises(RuntimeError):
        torch.vmap(layer)(x)
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda x: layer(x).sum())(x)
    with fwad.dual_level(), pytest.raises(NotImplementedError):
        layer(fwad.make_dual(x, torch.ones_like(x)))


def test_host_tensors_are_refused(layer):
    import blockwise_int8_linear_amd as pkg
    layer.eval()
    with torch.no_grad():
        layer(torch.randn(1, 192, device=DEV))
        with pytest.raises(AssertionError):
            layer(torch.randn(1, 192))
    codes, scales = pkg.quantize_block_rowwise(layer.weight.detach())
    with pytest.raises(AssertionError):
        pkg.dequantize_block_rowwise(codes, scales.cpu())
    with pytest.raises(AssertionError):
        pkg.int8_matmul_block64_rowwise_dequantize(codes, codes.t(), scales.cpu(), scales)
