"""The native host path (csrc/torch_ops.cpp) against the Python functions it stands in for."""
import pytest
import torch

from ipex_llm.ggml.quantize import ggml_tensor_qtype as Q
from ipex_llm.transformers.low_bit_linear import (FP4Params, batch_forward, dequantize_rows, forward_new, mlp_forward_xpu,
                                                  use_batch_forward)
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


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,numel", [(torch.float16, (4 << 20) // 2 + 1), (torch.uint8, (8 << 20) + 3), (torch.float32, 3 << 20), (torch.bfloat16, 9 << 20)])
def test_large_copies_through_pinned_chunks(dtype, numel):
    t = torch.randint(0, 200, (numel + 5,)).to(dtype)[5:]                        # not at the start of its storage
    up = ops.upload(t, 0)
    assert up.device.type == "cuda" and up.dtype == dtype and torch.equal(up, t.cuda())
    down = ops.download(up)
    assert down.device.type == "cpu" and torch.equal(down, t)
    assert ops.upload(t[:100], 0) is None and ops.upload(t[::2], 0) is None and ops.upload(up, 0) is None and ops.download(t) is None


@pytest.mark.gpu
@pytest.mark.parametrize("qname", ["sym_int4", "asym_int4", "sym_int8", "nf4", "fp8_e4m3"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,k", [(3, 128), (48, 640), (2048, 1152)])
def test_half_precision_sources_quantize_as_their_float32_values(qname, dtype, n, k):
    torch.manual_seed(n)
    w = (torch.randn(n, k) * 0.02).to(dtype)
    def blob(t, device):
        return FP4Params(t, qtype=Q[qname]).to(device).data.view(torch.uint8)
    want, tiled = blob(w.float(), "cpu"), blob(w.float().cuda(), "cuda")
    for src in (w, w.t().contiguous().t()):                                       # contiguous, and not
        assert torch.equal(blob(src, "cpu"), want)
        assert torch.equal(blob(src, "cuda"), tiled) and torch.equal(blob(src.cuda(), "cuda"), tiled)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("offset", [1, 3, 4])
def test_weights_that_start_between_16_byte_boundaries(dtype, offset):
    flat = torch.randn(offset + 48 * 256, device="cuda").to(dtype)
    view = flat[offset:].view(48, 256)
    for place in (lambda p: p.to("cuda"), lambda p: p.quantize("cpu")):
        got, want = (place(FP4Params(w, qtype=Q["sym_int4"])).data for w in (view, view.clone()))
        assert torch.equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("qname", ["sym_int4", "asym_int4", "sym_int8", "nf4", "fp8_e4m3"])
@pytest.mark.parametrize("m,n,k", [(1, 64, 256), (2, 64, 128), (48, 80, 128), (49, 64, 384), (49, 80, 256), (64, 64, 256), (65, 64, 256)])
def test_float32_batches_follow_use_batch_forward(qname, m, n, k):
    torch.manual_seed(m + n)
    w, x = FP4Params(torch.randn(n, k) * 0.02, qtype=Q[qname]).to("cuda"), torch.randn(m, k, device="cuda")
    stays = m == 1 or use_batch_forward(x, Q[qname], n)
    want = (batch_forward if stays else forward_new)(x, w.data, Q[qname], n, layout=w.blob_layout)
    assert torch.equal(ops.linear(x, w, None, Q[qname], n, True), want)
    assert torch.equal(ops.linear(x, w, None, Q[qname], n, False), batch_forward(x, w.data, Q[qname], n, layout=w.blob_layout))


@pytest.mark.gpu
@pytest.mark.parametrize("qname", ["sym_int4", "nf4", "fp8_e4m3"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,act", [(1, 0), (6, 1), (40, 0), (70, 1)])
def test_native_gated_equals_mlp_forward_xpu(qname, dtype, m, act):
    torch.manual_seed(m)
    wg, wu = (FP4Params(torch.randn(272, 256) * 0.05, qtype=Q[qname]).to("cuda") for _ in range(2))
    x = torch.randn(1, m, 512, device="cuda").to(dtype)[..., :256]                # three dimensions, rows that are not contiguous
    got = ops.gated(x, wg, wu, Q[qname], 272, act)
    want = mlp_forward_xpu(x.contiguous().view(m, 256), wg.data, wu.data, m, 256, 272, act, Q[qname])
    assert got.shape == (1, m, 272) and got.dtype == dtype and torch.equal(got[0], want)
    assert ops.gated(x.float(), wg, wu, Q[qname], 272, act) is None
    assert ops.gated(x, wg, FP4Params(torch.randn(272, 384), qtype=Q[qname]).to("cuda"), Q[qname], 272, act) is None


@pytest.mark.gpu
@pytest.mark.parametrize("qname", ["sym_int4", "asym_int4", "sym_int8", "nf4", "fp8_e4m3"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,k", [(48, 256), (37, 128)])
def test_native_embedding_equals_the_python_steps(qname, dtype, n, k):
    torch.manual_seed(n)
    table, like = FP4Params(torch.randn(n, k), qtype=Q[qname]).to("cuda"), torch.empty(0, dtype=dtype, device="cuda")
    ids = torch.randint(0, n, (3, 8), device="cuda")[:, ::2]
    got = ops.embedding(ids, table, Q[qname], n, k, like)
    want = dequantize_rows(ids.contiguous(), table.data, Q[qname], k, n, layout=table.blob_layout).to(dtype)
    assert got.shape == (3, 4, k) and got.dtype == dtype and torch.equal(got, want)
    assert ops.embedding(ids.int(), table, Q[qname], n, k, like) is None and ops.embedding(ids, table, Q[qname], n + 1, k, like) is None
