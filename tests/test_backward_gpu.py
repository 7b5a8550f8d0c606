"""The gradient that flows on below a low-bit linear, from the packed weight."""
import pytest
import torch

from gpu_util import ALL, DT, NAMES, dev_dequantize, dev_quantize, ggml, stream, weights

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
