"""The mixture-of-experts block as one call (csrc/moe.hip) against the loop over its experts' layers."""
import pytest
import torch
from torch import nn

from ipex_llm.ggml.quantize import ggml_tensor_qtype as Q
from ipex_llm.transformers.low_bit_linear import FP4Params, LowBitLinear, dequant
from ipex_llm.transformers.native_ops import ops
from ipex_llm.transformers.moe import ExpertWeights, LowBitExperts, moe_ffn_grouped, moe_ffn_reference, route_top_k

pytestmark = pytest.mark.gpu


def _layers(n_exp, n, k, qtype):
    with torch.device("meta"):
        layers = nn.ModuleList([LowBitLinear(k, n, qtype, bias=False) for _ in range(n_exp)])
    for layer in layers:
        layer._parameters["weight"] = FP4Params(torch.randn(n, k, device="cuda") * 0.05, qtype=qtype).to("cuda")
    return layers.eval()


def _block(n_exp, hidden, inter, qtype):
    with torch.device("meta"):
        block = LowBitExperts(n_exp, hidden, inter, qtype, nn.SiLU())
    block.gate, block.up = _layers(n_exp, inter, hidden, qtype), _layers(n_exp, inter, hidden, qtype)
    block.down = _layers(n_exp, hidden, inter, qtype)
    return block.eval()


def _tables(block):
    return [ExpertWeights(list(layers)) for layers in (block.gate, block.up, block.down)]


def _close(got, want):
    """Within what fp16 sums in another order and one rounding more or less differ by."""
    assert got.dtype == want.dtype and got.shape == want.shape
    assert (got.float() - want.float()).abs().max() <= 4e-3 * want.float().abs().max()


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


@pytest.mark.parametrize("tokens,top_k,n_exp,hidden", [(85, 3, 8, 128), (86, 3, 8, 2048), (1024, 4, 16, 256), (1025, 4, 16, 256), (683, 3, 512, 128),
                                                       (9, 2, 4, 4224)])
def test_pairs_around_the_rounds_of_their_counting(tokens, top_k, n_exp, hidden):
    """255 and 258 pairs, 4096 and beyond (the two launches), 2049, 512 experts; rows of 16 pieces up to more than the 512 held; two
    pairs without an expert."""
    torch.manual_seed(tokens)
    block = _block(n_exp, hidden, 128, Q["sym_int4"])
    x = torch.randn(tokens, hidden, device="cuda").half()
    weight, index = torch.topk(torch.softmax(torch.randn(tokens, n_exp, device="cuda"), -1), top_k, dim=-1)
    index[0, 0], index[tokens - 1, top_k - 1] = -1, n_exp
    got = block(x, index, weight.half())
    weight[0, 0], index[0, 0], weight[tokens - 1, top_k - 1], index[tokens - 1, top_k - 1] = 0, 0, 0, 0
    _close(got, block._loop(x, index, weight.half()))


@pytest.mark.parametrize("top_k", [1, 2, 3, 4, 5, 7, 8, 9])
def test_experts_per_token_summed_in_fours_and_a_rest(top_k):
    """Pairs without an expert at the start, at the end, and all of one token: its row is zero."""
    torch.manual_seed(top_k)
    block = _block(10, 256, 128, Q["sym_int8"])
    x = torch.randn(21, 256, device="cuda").half()
    weight, index = torch.topk(torch.softmax(torch.randn(21, 10, device="cuda"), -1), top_k, dim=-1)
    index[0, 0], index[20, top_k - 1], index[7] = -1, 10, -1
    got = block(x, index, weight.half())
    weight[0, 0], index[0, 0], weight[20, top_k - 1], index[20, top_k - 1], weight[7], index[7] = 0, 0, 0, 0, 0, 0
    _close(got, block._loop(x, index, weight.half()))
    assert (got[7] == 0).all()


def test_experts_follow_a_weight_that_was_replaced():
    torch.manual_seed(5)
    block = _block(4, 128, 256, Q["sym_int4"])
    x, index = torch.randn(9, 128, device="cuda").half(), torch.randint(0, 4, (9, 2), device="cuda")
    weight = torch.rand(9, 2, device="cuda").half()
    block(x, index, weight)
    block.down[2]._parameters["weight"] = FP4Params(torch.randn(128, 256, device="cuda") * 0.05, qtype=Q["sym_int4"]).to("cuda")
    got, want = block(x, index, weight), block._loop(x, index, weight)
    assert (got.float() - want.float()).abs().max() <= 4e-3 * want.float().abs().max()


@pytest.mark.parametrize("qname,down", [("sym_int4", "sym_int8"), ("sym_int8", "sym_int4"), ("fp8_e4m3", "nf4")])
def test_down_weights_of_another_format(qname, down):
    torch.manual_seed(6)
    block = _block(4, 128, 256, Q[qname])
    block.down = _layers(4, 128, 256, Q[down])
    x, logits = torch.randn(9, 128, device="cuda").half(), torch.randn(9, 4, device="cuda")
    weight, index = route_top_k(logits)
    want = block._loop(x, index, weight)
    _close(block(x, index, weight), want)
    _close(moe_ffn_grouped(x, logits, *_tables(block)), want)
    index[2, 0], weight[2, 0] = 4, float("nan")                                   # a pair without an expert counts nothing
    got = block(x, index, weight)
    weight[2, 0], index[2, 0] = 0, 0
    _close(got, block._loop(x, index, weight))
    with pytest.raises(RuntimeError, match="fit together"):
        block(x[:1], index[:1], weight[:1])


@pytest.mark.parametrize("table,n_exp,n,k", [(1, 4, 384, 128), (1, 4, 256, 256), (1, 3, 256, 128), (2, 4, 128, 128), (2, 4, 256, 256),
                                             (2, 3, 128, 256)])
def test_tables_that_do_not_fit_together_are_refused(table, n_exp, n, k):
    block = _block(4, 128, 256, Q["sym_int4"])
    tables = _tables(block)
    tables[table] = ExpertWeights(list(_layers(n_exp, n, k, Q["sym_int4"])))
    x, logits = torch.randn(9, 128, device="cuda").half(), torch.randn(9, 4, device="cuda")
    with pytest.raises(RuntimeError, match="fit together"):
        moe_ffn_grouped(x, logits, *tables)
    block.__dict__["_tables"] = tuple(tables)                                     # as after layers were replaced
    weight, index = route_top_k(logits)
    for tokens in (1, 9):
        with pytest.raises(RuntimeError, match="fit together"):
            block(x[:tokens], index[:tokens], weight[:tokens])
    g, u, d = (t.ptrs for t in _tables(block))
    bad = (g, u[:3], d) if table == 1 else (g, u, d.cpu())
    assert ops.experts(x, index, weight, *bad, Q["sym_int4"], 128, 256, 0) is None


@pytest.mark.parametrize("tokens", [1, 3, 9])
def test_indices_of_other_integer_types_take_the_same_call(tokens):
    torch.manual_seed(tokens)
    block = _block(4, 128, 256, Q["sym_int4"])
    x, index = torch.randn(tokens, 128, device="cuda").half(), torch.randint(0, 4, (tokens, 2), device="cuda")
    weight = torch.rand(tokens, 2, device="cuda").half()
    want = block(x, index, weight)
    for dtype in (torch.int32, torch.int16, torch.uint8):
        assert torch.equal(block(x, index.to(dtype), weight), want)
    index32, graph = index.int(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):                                                 # nothing in it waits for the host
        got = block(x, index32, weight)
    for _ in range(3):
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)
        x.neg_()
        want = block(x, index, weight)


def test_calls_beyond_the_native_one():
    torch.manual_seed(7)
    block = _block(70, 128, 128, Q["sym_int4"])
    tables = _tables(block)
    x, logits = torch.randn(5, 128, device="cuda").half(), torch.randn(5, 70, device="cuda")
    assert moe_ffn_grouped(x[:0], logits[:0], *tables).shape == (0, 128)
    for top_k in (64, 66):                                                        # at most 64 in the native call
        weight, index = route_top_k(logits, top_k)
        want = block._loop(x, index, weight)
        _close(moe_ffn_grouped(x, logits, *tables, top_k=top_k), want)
        for tokens in (1, 5):
            _close(block(x[:tokens], index[:tokens], weight[:tokens]), want[:tokens])
    weight, index = route_top_k(logits)
    for tokens in (1, 5):                                                         # routing that stayed on the host
        want = block(x[:tokens], index[:tokens], weight[:tokens])
        _close(block(x[:tokens], index[:tokens].cpu(), weight[:tokens].cpu()), want)
    with pytest.raises(RuntimeError):
        block(x, index, weight[:4])
    # more experts than the native call sorts: the same layers again and again
    g, u, d = ([layers[e % 70] for e in range(4100)] for layers in (block.gate, block.up, block.down))
    logits = torch.randn(5, 4100, device="cuda")
    _close(moe_ffn_grouped(x, logits, ExpertWeights(g), ExpertWeights(u), ExpertWeights(d)), moe_ffn_reference(x, logits, g, u, d))


def test_routing_weights_get_their_gradient():
    torch.manual_seed(8)
    block = _block(4, 128, 256, Q["sym_int4"])
    x, logits = torch.randn(9, 128, device="cuda").half(), torch.randn(9, 4, device="cuda").requires_grad_(True)
    weight, index = route_top_k(logits)
    index[2, 0] = 4                                                               # a pair without an expert
    weight = weight.detach().requires_grad_(True)
    y = block(x, index, weight)
    with torch.no_grad():
        one = [block(x, index, torch.nn.functional.one_hot(torch.full((9,), j, device="cuda"), 2).half()) for j in range(2)]
    _close(y.detach(), block(x, index, weight.detach()))
    (grad,) = torch.autograd.grad(y.float().sum(), weight)
    want = torch.stack([t.float().sum(-1) for t in one], -1)
    assert grad[2, 0] == 0 and (grad - want).abs().max() <= 4e-3 * want.abs().max()
    (grad,) = torch.autograd.grad(moe_ffn_grouped(x, logits, *_tables(block)).float().pow(2).sum(), logits)
    assert torch.isfinite(grad).all() and grad.abs().max() > 0
    with torch.no_grad():
        assert not block(x, index, weight).requires_grad
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(weight.detach(), torch.ones_like(weight))
        assert torch.autograd.forward_ad.unpack_dual(block(x, index, dual)).tangent is not None


@pytest.mark.parametrize("qname", ["sym_int4", "asym_int4", "nf4", "sym_int8"])
@pytest.mark.parametrize("tokens", [1, 3])
def test_an_activation_that_overflows_meets_the_weights(qname, tokens):
    """One of an expert's intermediate values is beyond fp16: its column of the down weights decides what the results are."""
    torch.manual_seed(9)
    block = _block(4, 128, 256, Q[qname])
    for layers in (block.gate, block.up):
        for layer in layers:
            w = torch.rand(256, 128, device="cuda") * 0.02
            w[17] = 5.0
            layer._parameters["weight"] = FP4Params(w, qtype=Q[qname]).to("cuda")
    x = torch.rand(tokens, 128, device="cuda").half() + 1                         # gate and up are 900 and more there, 3 at most elsewhere
    index, weight = torch.arange(tokens, device="cuda")[:, None], torch.full((tokens, 1), 0.5, device="cuda")
    y = block(x, index, weight).float().cpu()
    for t in range(tokens):
        down = block.down[t].weight
        col = dequant(torch.empty(0, device="cuda"), down.data, Q[qname], shape=(128, 256)).view(128, 256)[:, 17].cpu()
        assert torch.equal(y[t].isnan(), col == 0) and torch.equal(y[t] == float("inf"), col > 0) and torch.equal(y[t] == -float("inf"), col < 0)
