"""The mixture-of-experts block as one call (csrc/moe.hip) against the loop over its experts' layers."""
import pytest
import torch
from torch import nn

from ipex_llm.ggml.quantize import ggml_tensor_qtype as Q
from ipex_llm.transformers.low_bit_linear import FP4Params
from ipex_llm.transformers.moe import LowBitExperts

pytestmark = pytest.mark.gpu


def _block(n_exp, hidden, inter, qtype):
    with torch.device("meta"):
        block = LowBitExperts(n_exp, hidden, inter, qtype, nn.SiLU())
    for layers, n, k in ((block.gate, inter, hidden), (block.up, inter, hidden), (block.down, hidden, inter)):
        for layer in layers:
            layer._parameters["weight"] = FP4Params(torch.randn(n, k, device="cuda") * 0.05, qtype=qtype).to("cuda")
    return block.eval()


# pairs around a wave, a workgroup and several rounds of the sort; experts around a wave, beyond it, and beyond 512
@pytest.mark.parametrize("qname,dtype", [("sym_int4", torch.float16), ("fp8_e4m3", torch.bfloat16)])
@pytest.mark.parametrize("tokens,top_k,n_exp", [(1, 4, 60), (2, 1, 4), (3, 2, 65), (8, 4, 8), (37, 3, 5), (16, 4, 64), (512, 2, 8),
                                                (700, 4, 60), (50, 2, 600)])
@pytest.mark.parametrize("wdtype", [None, torch.float32])
def test_experts_equal_the_loop_over_their_layers(qname, dtype, tokens, top_k, n_exp, wdtype):
    torch.manual_seed(tokens + n_exp)
    block = _block(n_exp, 256, 384, Q[qname])
    x = torch.randn(tokens, 256, device="cuda").to(dtype)
    # an uneven choice: some experts get no rows
    logits = torch.randn(tokens, n_exp, device="cuda") + 2 * torch.randn(1, n_exp, device="cuda")
    weight, index = torch.topk(torch.softmax(logits, -1), top_k, dim=-1)
    weight = weight.to(wdtype or dtype)
    got, want = block(x, index, weight), block._loop(x, index, weight)
    assert got.dtype == dtype and got.shape == want.shape
    tol = 4e-3 if dtype == torch.float16 else 2e-2                       # the loop rounds the activation and every sum
    assert (got.float() - want.float()).abs().max() <= tol * want.float().abs().max()
    if tokens > 1:
        # a pair without an expert counts nothing
        index[1, 0] = n_exp
        weight[1, 0] = float("nan")
        again = block(x, index, weight)
        weight[1, 0], index[1, 0] = 0, 0
        want = block._loop(x, index, weight)
        assert (again.float() - want.float()).abs().max() <= tol * want.float().abs().max()


def test_experts_follow_a_weight_that_was_replaced():
    torch.manual_seed(5)
    block = _block(4, 128, 256, Q["sym_int4"])
    x, index = torch.randn(9, 128, device="cuda").half(), torch.randint(0, 4, (9, 2), device="cuda")
    weight = torch.rand(9, 2, device="cuda").half()
    block(x, index, weight)
    block.down[2]._parameters["weight"] = FP4Params(torch.randn(128, 256, device="cuda") * 0.05, qtype=Q["sym_int4"]).to("cuda")
    got, want = block(x, index, weight), block._loop(x, index, weight)
    assert (got.float() - want.float()).abs().max() <= 4e-3 * want.float().abs().max()
