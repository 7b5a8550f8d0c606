"""The gradient that flows on below a low-bit linear: the kernel that reads the packed weight, and the layer around it."""
import pytest
import torch

from gpu_util import ALL, DT, NAMES, dev_dequantize, dev_quantize, ggml, stream, weights
from ipex_llm.transformers.low_bit_linear import FP4Params, LowBitLinear, MatMulLowBit

pytestmark = pytest.mark.gpu
TILED = ggml.LAYOUT_TILED


def close(got, grad, w, dtype):
    """One rounding of the result, fp32 sums of n terms, weights that are the 16-bit ones of dev_dequantize (asym_int4: q * d + m
    may round from fp32 or from the exact value)."""
    want, size = grad.double() @ w.double(), grad.float().abs() @ w.float().abs()
    eps = torch.finfo(dtype).eps
    bound = want.abs() * eps / 2 + size * (grad.shape[0 if grad.dim() == 1 else -1] * 2.0 ** -24 + 2.0 ** -24) + torch.finfo(dtype).smallest_normal
    return ((got.double() - want).abs() <= bound).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("m,n,k", [(1, 16, 128), (33, 64, 128), (64, 80, 256), (65, 112, 384), (200, 832, 256), (130, 1200, 640),
                                   (2100, 144, 1024), (8193, 48, 128)])
@pytest.mark.parametrize("qtype", ALL, ids=NAMES.values())
def test_kernel(qtype, m, n, k, dtype):
    """Last steps of 16, 32, 48 and 64 weight rows, one step (a group of waves without any), odd and even numbers of them up to
    nineteen, row tiles of 64 and of 128 with rows past M; rows of g that hold an infinity."""
    blob = dev_quantize(weights(5, (n, k)), qtype, TILED)
    gen = torch.Generator().manual_seed(m)
    grad = torch.randn((m, n), generator=gen).to(dtype).cuda()
    out = torch.full((m + 1, k), float("nan"), dtype=dtype, device="cuda")
    ggml.lowbit_backward(grad.data_ptr(), blob.data_ptr(), out.data_ptr(), qtype, DT[dtype], m, n, k, stream())
    w = dev_dequantize(blob, qtype, n, k, TILED, dtype)
    assert torch.isnan(out[m]).all()
    assert close(out[:m], grad, w, dtype)
    grad[0, n - 1] = float("inf")                           # next to the columns past N of a last step
    ggml.lowbit_backward(grad.data_ptr(), blob.data_ptr(), out.data_ptr(), qtype, DT[dtype], m, n, k, stream())
    want = grad[:1].float().cpu() @ w.float().cpu()
    assert torch.equal(out[:1].float().cpu().isnan(), want.isnan()) and torch.equal(out[:1].float().cpu().isinf(), want.isinf())
    assert m == 1 or close(out[1:m], grad[1:], w, dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("m,n,k", [(1030, 1200, 2048), (2100, 1616, 1024), (1024, 1664, 2176)])
@pytest.mark.parametrize("qtype", ALL, ids=NAMES.values())
def test_kernel_of_128_rows_over_many_steps(qtype, m, n, k, dtype):
    """Row tiles of 128 (more than 256 of 64), each group of waves past its loop's period of six: 19 and 26 steps, a last one of 48
    and of 16 weight rows and whole ones."""
    assert (m + 63) // 64 * (k // 128) > 256
    test_kernel(qtype, m, n, k, dtype)


def layer_of(qtype, n, k, bias=None):
    with torch.device("meta"):
        layer = LowBitLinear(k, n, qtype, bias=bias is not None)
    layer._parameters["weight"] = FP4Params(torch.from_numpy(weights(9, (n, k))), qtype=qtype).to("cuda")
    if bias is not None:
        layer._parameters["bias"] = torch.nn.Parameter(bias, requires_grad=False)
    return layer.train()


@pytest.mark.parametrize("m,n,k", [(100, 1024, 2560), (100, 4096, 512), (70, 528, 1056)], ids=["packed", "dense", "row-major"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
def test_layer_in_training(m, n, k, dtype):
    """Both ways of the gradient and both layouts, against the autograd function in Python; x and its gradient of other strides."""
    gen = torch.Generator().manual_seed(3)
    layer = layer_of(2, n, k, torch.randn(n, generator=gen).to(dtype).cuda())
    layout = layer.weight.blob_layout
    assert ggml.lowbit_backward_applies(2, layout, DT[dtype], m, n, k) == (layout == TILED and n < 2 * k)
    x = torch.randn((2, k, m // 2), generator=gen).to(dtype).cuda().transpose(1, 2).requires_grad_(True)
    y = layer(x)
    assert y.grad_fn.name() == "MatMulLowBitBackward" and y.shape == (2, m // 2, n)
    with torch.inference_mode():
        assert torch.equal(y, layer.eval()(x.detach()))
    layer.train()
    w = dev_dequantize(layer.weight.data.view(torch.uint8), 2, n, k, layout, dtype)
    grad = torch.randn((2, n, m // 2), generator=gen).to(dtype).cuda().transpose(1, 2)
    for _ in range(2):                                       # nothing is freed by the first backward
        (gx,) = torch.autograd.grad(y, x, grad)
        assert gx.shape == x.shape and close(gx.reshape(m, k), grad.reshape(m, n), w, dtype)
    (gs,) = torch.autograd.grad(y.sum(), x)                  # a gradient of strides 0
    assert close(gs.reshape(m, k), torch.ones((m, n), dtype=dtype, device="cuda"), w, dtype)
    product = MatMulLowBit.apply(x.detach().reshape(m, k).requires_grad_(True), layer.weight, n).view(y.shape)
    eps = torch.finfo(dtype).eps                             # that rounds the product and the sum with the bias, the layer the sum
    assert ((product + layer.bias - y).abs() <= eps * (product.abs() / 2 + y.abs())).all()


@pytest.mark.parametrize("m,n,k", [(24, 64, 128), (100, 1024, 2560)], ids=["dense", "packed"])
def test_derivatives_that_the_node_leaves_to_operators(m, n, k):
    """A second derivative, a batch of gradients, tangents and a saved-tensor hook, as MatMulLowBit has them, at sizes where a plain
    gradient comes from the packed weight and where it does not."""
    assert ggml.lowbit_backward_applies(2, TILED, DT[torch.float16], m, n, k) == (n > 64)
    layer = layer_of(2, n, k)
    w = dev_dequantize(layer.weight.data.view(torch.uint8), 2, n, k, TILED, torch.float16)
    x = torch.randn((m, k), device="cuda").half().requires_grad_(True)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: pytest.fail("nothing is saved"), lambda t: t):
        y = layer(x)
    grad = torch.randn((m, n), device="cuda").half().requires_grad_(True)
    (gx,) = torch.autograd.grad(y, x, grad, create_graph=True)
    v = torch.randn((m, k), device="cuda").half()
    (gg,) = torch.autograd.grad(gx, grad, v, retain_graph=True)
    assert close(gg, v, w.t(), torch.float16)
    batch = torch.randn((3, m, n), device="cuda").half()
    (gb,) = torch.autograd.grad(y, x, batch, is_grads_batched=True, retain_graph=True)
    for i in range(3):
        assert close(gb[i], batch[i], w, torch.float16)
    with torch.autograd.forward_ad.dual_level():
        (gt,) = torch.autograd.grad(y, x, torch.autograd.forward_ad.make_dual(batch[0], batch[1]))
        primal, tangent = torch.autograd.forward_ad.unpack_dual(gt)
        assert close(primal, batch[0], w, torch.float16) and close(tangent, batch[1], w, torch.float16)
        dual = torch.autograd.forward_ad.make_dual(x, torch.ones_like(x))
        with pytest.raises(RuntimeError):
            layer(dual)
    with torch.no_grad():
        assert not layer(x).requires_grad


class LeavesOut(torch.autograd.Function):
    @staticmethod
    def forward(ctx, y):
        return y.clone()

    @staticmethod
    def backward(ctx, grad):
        return None


@pytest.mark.parametrize("m,n,k", [(24, 64, 128), (100, 1024, 2560)], ids=["dense", "packed"])
def test_a_gradient_that_is_left_out_counts_as_zeros(m, n, k):
    """As MatMulLowBit, an autograd function in Python, is given it."""
    layer = layer_of(2, n, k)
    x = torch.randn((2, m // 2, k), device="cuda").half().requires_grad_(True)
    for product in (layer, lambda t: MatMulLowBit.apply(t.view(m, k), layer.weight, n)):
        (gx,) = torch.autograd.grad(LeavesOut.apply(product(x)).sum(), x)
        assert gx.shape == x.shape and gx.dtype == x.dtype and not gx.any()


class Operators(torch.utils._python_dispatch.TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.seen = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.seen.append(func._schema.name)
        return func(*args, **(kwargs or {}))


def test_transforms_and_modes_get_what_the_autograd_function_gives():
    """A transform that MatMulLowBit refuses is refused, a dispatch mode sees the operators of the backward, and a trace holds the
    layer: at a size where a plain gradient comes from the packed weight."""
    m, n, k = 100, 1024, 2560
    assert ggml.lowbit_backward_applies(2, TILED, DT[torch.float16], m, n, k)
    layer = layer_of(2, n, k)
    w = dev_dequantize(layer.weight.data.view(torch.uint8), 2, n, k, TILED, torch.float16)
    x = torch.randn((m, k), device="cuda").half().requires_grad_(True)
    grad = torch.randn((m, n), device="cuda").half()
    for product in (layer, lambda t: MatMulLowBit.apply(t, layer.weight, n)):
        with pytest.raises(RuntimeError):
            torch.func.grad(lambda t: product(t).sum())(x)
        with pytest.raises(RuntimeError):
            torch.func.vmap(product)(x.view(4, m // 4, k))
        with Operators() as mode:
            (gx,) = torch.autograd.grad(product(x), x, grad)
        assert "aten::mm" in mode.seen and close(gx, grad, w, torch.float16)
    traced = torch.jit.trace(layer, x, check_trace=False)
    assert torch.equal(traced(x), layer(x))


@pytest.mark.parametrize("m,n,k,rows", [(24, 4096, 1024, 64), (65, 2992, 1152, 64), (139, 4096, 2304, 64), (300, 6160, 1152, 64), (500, 8208, 2048, 128)])
@pytest.mark.parametrize("qtype", ALL, ids=NAMES.values())
def test_shared_walks(qtype, m, n, k, rows):
    """Several workgroups on a tile's walk along N: last splits of other lengths than the first, a last step of 16 and 48 rows, row tiles
    with rows past M; no more of the workspace is written than was asked for, and with half of it the answer is as good."""
    dtype = torch.bfloat16 if qtype in (3, 15) else torch.float16
    need = ggml.lowbit_backward_workspace_bytes(qtype, m, n, k)
    per_split = -(-m // rows) * rows * k * 4
    assert need >= 2 * per_split and need % per_split == 0 and need // per_split * (per_split // (rows * 512)) <= 256
    blob = dev_quantize(weights(5, (n, k)), qtype, TILED)
    grad = torch.randn((m, n), generator=torch.Generator().manual_seed(m)).to(dtype).cuda()
    w = dev_dequantize(blob, qtype, n, k, TILED, dtype)
    for size in (need, need // 2 // 16 * 16, 0):
        ws = torch.full((need + 64,), 255, dtype=torch.uint8, device="cuda")
        out = torch.full((m + 1, k), float("nan"), dtype=dtype, device="cuda")
        ggml.lowbit_backward_ws(grad.data_ptr(), blob.data_ptr(), out.data_ptr(), qtype, DT[dtype], m, n, k, ws.data_ptr(), size, stream())
        assert torch.isnan(out[m]).all() and close(out[:m], grad, w, dtype)
        assert (ws[size:] == 255).all()
