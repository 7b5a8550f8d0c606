"""The native host path (csrc/torch_ops.cpp) against the Python functions it stands in for."""
import pytest
import torch

from ipex_llm.ggml.quantize import ggml_tensor_qtype as Q
from ipex_llm.transformers.low_bit_linear import FP4Params, batch_forward, forward_new
from ipex_llm.transformers.native_ops import ops


def test_anything_but_the_plain_case_is_left_to_python():
    x, w = torch.zeros(2, 64), torch.zeros(72, dtype=torch.uint8)
    assert ops.linear(x, w, None, Q["sym_int4"], 2, True) is None                 # not on the GPU
    assert ops.gated(x, w, w, Q["sym_int4"], 2, 0) is None
    assert ops.embedding(torch.zeros(3, dtype=torch.int64), w, Q["sym_int4"], 2, 64, x) is None
    with pytest.raises(TypeError):
        ops.linear(x, w, None, "sym_int4", 2, True)


@pytest.mark.gpu
@pytest.mark.parametrize("qname", ["sym_int4", "nf4"])
@pytest.mark.parametrize("m,n,k", [(1, 16, 128), (17, 37, 192), (48, 64, 256), (65, 64, 256)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_native_linear_equals_the_python_functions(qname, m, n, k, dtype):
    torch.manual_seed(m + n)
    w = FP4Params(torch.randn(n, k) * 0.02, qtype=Q[qname]).to("cuda")
    x = torch.randn(m, 2 * k, device="cuda").to(dtype)[:, :k]                     # rows that are not contiguous
    stays = dtype == torch.float32 and (m == 1 or (qname == "sym_int4" and m <= 64 and k % 128 == 0 and m != 65))
    want = (batch_forward if stays else forward_new)(x, w.data, Q[qname], n, layout=w.blob_layout)
    got = ops.linear(x, w, None, Q[qname], n, True)
    assert got.dtype == dtype and torch.equal(got, want)
    assert ops.linear(x, w, None, Q[qname], n + 1, True) is None                  # a weight of another size
