"""The work that users of this package have it do, as cases that can be timed.

Every case goes through the modules a converted model holds (LowBitLinear, the fused gated MLP, LowBitEmbedding,
LowBitExperts) or through optimize_model.  Weights are N(0, 0.02) and activations N(0, 1) with a few channels of
large magnitude, as language models have them; everything is made from the seed.

Kinds of case:
  linear   one LowBitLinear at inference, any number of rows, 16-bit or float32 activations, any shape that converts
  step     what one decoding step of a converted model calls: token embedding, per layer the merged q/k/v, the output
           projection and the gated MLP, then the head.  "graph": the same calls captured once in a HIP graph and
           replayed, as a server does
  layer    the linears of one decoder layer on a prompt
  train    forward and backward of a LowBitLinear below trained parameters (adapter finetuning)
  experts  the experts of a mixture-of-experts block
  load     optimize_model on a dense layer in host memory, then .to("cuda"): what loading a checkpoint does per layer
"""
import math
import os
import sys

import torch
from torch import nn

sys.path.insert(0, os.path.abspath("ipex-llm_amd"))        # the package lives beside this folder, in the working directory

import ipex_llm.ggml.model.llama.llama_cpp as ggml  # noqa: E402
from ipex_llm import optimize_model  # noqa: E402
from ipex_llm.ggml.quantize import ggml_tensor_qtype  # noqa: E402
from ipex_llm.transformers.embedding import LowBitEmbedding  # noqa: E402
from ipex_llm.transformers.low_bit_linear import FP4Params, LowBitLinear  # noqa: E402
from ipex_llm.transformers.models.common import mlp_silu_forward  # noqa: E402
from ipex_llm.transformers.moe import LowBitExperts  # noqa: E402

FORMATS = ("sym_int4", "asym_int4", "sym_int8", "nf4", "fp8_e4m3")
BATCH_F32 = ("sym_int4", "asym_int4", "fp8_e4m3")      # formats whose small batches stay float32 with float32 activations
DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32}
MOST_FLOPS = 8.2e11                                    # just below the largest listed case
MOST_BYTES = 1.8e9


def listed():
    return [
        # chat with one user: one projection of one new token; the launch and the Python around it count
        dict(name="decode_linear", kind="linear", qtype="sym_int4", dtype="float16", m=1, n=4096, k=4096, bias=False),
        # the same user, server with captured graphs: 16 layers stream 1.8 GB of weights for one token
        dict(name="decode_graph", kind="step", qtype="sym_int4", dtype="float16", m=1, layers=16, hidden=4096,
             kv=4096, inter=11008, vocab=0, graph=True),
        # eight users decoding together, eager; the vocabulary got three added tokens, so the head has odd rows
        dict(name="decode_step_batch8", kind="step", qtype="asym_int4", dtype="bfloat16", m=8, layers=4, hidden=4096,
             kv=1024, inter=11008, vocab=32003, graph=False),
        # a serving batch of a few dozen sequences through the widest projection
        dict(name="serve_batch40", kind="linear", qtype="sym_int4", dtype="float16", m=40, n=11008, k=4096, bias=True),
        # a model loaded without a 16-bit dtype: activations are float32 all the way
        dict(name="float32_batch12", kind="linear", qtype="sym_int4", dtype="float32", m=12, n=4096, k=4096, bias=False),
        # in_features that are no multiple of 128 keep the row-major blob: a short prompt through such a layer
        dict(name="ragged_prompt", kind="linear", qtype="sym_int4", dtype="float16", m=333, n=3200, k=8640, bias=False),
        # a long prompt through one decoder layer
        dict(name="prefill_layer", kind="layer", qtype="sym_int4", dtype="float16", m=2048, hidden=4096, kv=4096,
             inter=11008),
        # a large model's widest layer, prompt of no round length
        dict(name="prefill_wide_nf4", kind="linear", qtype="nf4", dtype="bfloat16", m=1000, n=28672, k=8192, bias=False),
        # adapter finetuning: forward, and the gradient that flows on to the layer below
        dict(name="train_step_nf4", kind="train", qtype="nf4", dtype="bfloat16", m=1024, n=4096, k=4096),
        # a prompt through a mixture of eight experts
        dict(name="experts_prompt", kind="experts", qtype="fp8_e4m3", dtype="bfloat16", m=512, experts=8, top_k=2,
             hidden=4096, inter=14336),
        # one new token through many small experts
        dict(name="experts_decode", kind="experts", qtype="sym_int4", dtype="float16", m=1, experts=60, top_k=4,
             hidden=2048, inter=1408),
        # loading: a dense half-precision layer on the host becomes a low-bit layer on the GPU
        dict(name="load_layer", kind="load", qtype="sym_int4", dtype="float16", n=11008, k=4096),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _to(v, step):
    return max(step, v // step * step)


def draw(rng):
    while True:
        case = _draw(rng)
        need = work(case)
        if need["flops"] <= MOST_FLOPS and need["bytes"] <= MOST_BYTES:
            return case


def _draw(rng):
    kind = rng.choice(("linear", "linear", "linear", "linear", "step", "layer", "train", "experts", "load"))
    qtype, dtype = rng.choice(FORMATS), rng.choice(("float16", "bfloat16"))
    if kind == "linear":
        ragged = rng.random() < 0.25
        n, k = _log(rng, 512, 28672), _to(_log(rng, 512, 28672), 128)
        if ragged and rng.random() < 0.5 and qtype != "fp8_e4m3":
            k += 64                                    # whole blocks, no whole tiles of 128 columns
            n = _to(n, 16)
        elif not ragged:
            n = _to(n, 16)
        m = _log(rng, 1, 512 if ragged else 2048)
        if rng.random() < 0.15:
            dtype, m = "float32", (min(m, 48) if qtype in BATCH_F32 and k % 128 == 0 else 1)
        return dict(kind=kind, qtype=qtype, dtype=dtype, m=m, n=n, k=k, bias=rng.random() < 0.3)
    hidden = _to(_log(rng, 1024, 8192), 128)
    inter = _to(int(hidden * rng.uniform(2.0, 3.6)), 128)
    kv = _to(hidden // rng.choice((1, 2, 4, 8)), 128)
    if kind == "step":
        return dict(kind=kind, qtype=qtype, dtype=dtype, m=_log(rng, 1, 16), layers=rng.randint(1, 12), hidden=hidden, kv=kv,
                    inter=inter, vocab=_log(rng, 8000, 64000), graph=rng.random() < 0.4)
    if kind == "layer":
        return dict(kind=kind, qtype=qtype, dtype=dtype, m=_log(rng, 24, 2048), hidden=hidden, kv=kv, inter=inter)
    if kind == "train":
        return dict(kind=kind, qtype=qtype, dtype=dtype, m=_log(rng, 64, 2048), n=_to(_log(rng, 1024, 14336), 16), k=hidden)
    if kind == "experts":
        return dict(kind=kind, qtype=qtype, dtype=dtype, m=_log(rng, 1, 600), experts=_log(rng, 4, 64), top_k=rng.randint(1, 4),
                    hidden=_to(_log(rng, 1024, 4096), 128), inter=_to(_log(rng, 512, 14336), 128))
    return dict(kind=kind, qtype=qtype, dtype=dtype, n=_log(rng, 256, 11008), k=_to(_log(rng, 512, 8192), 128))


# ------------------------------------------------------------------ inputs

class GatedMLP(nn.Module):
    """The gated MLP block as model code has it; its forward is the one that the conversion binds to such blocks."""

    def __init__(self, gate, up, down):
        super().__init__()
        self.gate_proj, self.up_proj, self.down_proj, self.act_fn = gate, up, down, nn.SiLU()

    def forward(self, x):
        return mlp_silu_forward(self, x)


class Maker:
    """Layers and activations of one case, made on the GPU from one generator."""

    def __init__(self, case, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed * 1000003 + 17)
        self.qtype, self.dtype = ggml_tensor_qtype[case["qtype"]], DTYPES[case["dtype"]]

    def dense(self, n, k, std=0.02):
        return torch.randn((n, k), generator=self.gen, device="cuda") * std

    def packed(self, n, k, std=0.02):
        return FP4Params(self.dense(n, k, std), qtype=self.qtype).to("cuda")

    def linear(self, n, k, bias=False, **more):
        with torch.device("meta"):
            layer = LowBitLinear(k, n, self.qtype, bias=bias, **more)
        layer._parameters["weight"] = self.packed(n, k)
        if bias:
            layer._parameters["bias"] = nn.Parameter(self.dense(1, n)[0].to(self.dtype), requires_grad=False)
        return layer.eval()

    def mlp(self, hidden, inter):
        return GatedMLP(self.linear(inter, hidden), self.linear(inter, hidden), self.linear(hidden, inter)).eval()

    def embedding(self, vocab, hidden):
        table = LowBitEmbedding(vocab, hidden, device="meta", dtype=self.dtype, qtype=self.qtype)
        table._parameters["qweight"] = self.packed(vocab, hidden, 1.0)
        return table.eval()

    def rows(self, *shape):
        x = torch.randn(shape, generator=self.gen, device="cuda")
        big = torch.randint(0, shape[-1], (max(1, shape[-1] // 512),), generator=self.gen, device="cuda")
        x[..., big] *= 8.0
        return x.to(self.dtype)


def _step_modules(make, case):
    hidden, kv, inter = case["hidden"], case["kv"], case["inter"]
    layers = [(make.linear(hidden + 2 * kv, hidden), make.linear(hidden, hidden), make.mlp(hidden, inter))
              for _ in range(case.get("layers", 1))]
    vocab = case.get("vocab", 0)
    return layers, (make.embedding(vocab, hidden), make.linear(vocab, hidden, optimize_lm_head=True)) if vocab else (None, None)


def _step(state):
    """Attention, norms and residuals are the model's own: q/k/v and the MLP read the embedded token, the output
    projection reads an attention result that is there."""
    embed, head = state["ends"]
    h = embed(state["ids"]) if embed is not None else state["x"]
    outs = [h] if embed is not None else []
    for qkv, o, mlp in state["layers"]:
        outs += [qkv(h), o(state["attn"]), mlp(h)]
    if head is not None:
        outs.append(head(h))
    return outs


def prepare(case, seed):
    make, kind = Maker(case, seed), case["kind"]
    if kind == "linear":
        return dict(kind=kind, layer=make.linear(case["n"], case["k"], case["bias"]), x=make.rows(case["m"], case["k"]))
    if kind in ("step", "layer"):
        layers, ends = _step_modules(make, case)
        shape = (case["m"], 1) if kind == "step" else (1, case["m"])
        state = dict(kind=kind, layers=layers, ends=ends, x=make.rows(*shape, case["hidden"]),
                     attn=make.rows(*shape, case["hidden"]))
        if ends[0] is not None:
            state["ids"] = torch.randint(0, case["vocab"], shape, generator=make.gen, device="cuda")
        if case.get("graph", False):
            with torch.inference_mode():
                side = torch.cuda.Stream()
                side.wait_stream(torch.cuda.current_stream())
                with torch.cuda.stream(side):
                    _step(state)
                torch.cuda.current_stream().wait_stream(side)
                state["graph"] = torch.cuda.CUDAGraph()
                with torch.cuda.graph(state["graph"]):
                    state["outs"] = _step(state)
        return state
    if kind == "train":
        layer = make.linear(case["n"], case["k"]).train()
        return dict(kind=kind, layer=layer, x=make.rows(case["m"], case["k"]).requires_grad_(True),
                    grad=make.rows(case["m"], case["n"]) * 0.01)
    if kind == "experts":
        hidden, inter, n_exp = case["hidden"], case["inter"], case["experts"]
        with torch.device("meta"):
            block = LowBitExperts(n_exp, hidden, inter, make.qtype, nn.SiLU())
        for e in range(n_exp):
            block.gate[e]._parameters["weight"] = make.packed(inter, hidden)
            block.up[e]._parameters["weight"] = make.packed(inter, hidden)
            block.down[e]._parameters["weight"] = make.packed(hidden, inter)
        # some experts are liked more than others
        logits = torch.randn((case["m"], n_exp), generator=make.gen, device="cuda") + \
            0.5 * torch.randn((1, n_exp), generator=make.gen, device="cuda")
        weights, index = torch.topk(torch.softmax(logits, -1), case["top_k"], dim=-1)
        return dict(kind=kind, block=block.eval(), x=make.rows(case["m"], hidden), index=index,
                    weights=(weights / weights.sum(-1, keepdim=True)).to(make.dtype))
    return dict(kind=kind, low_bit=case["qtype"], w=make.dense(case["n"], case["k"]).to(make.dtype).cpu())


# ------------------------------------------------------------------ one pass

def run(state):
    kind = state["kind"]
    if kind == "train":
        y = state["layer"](state["x"])
        (gx,) = torch.autograd.grad(y, state["x"], state["grad"])
        return [y.detach(), gx]
    with torch.inference_mode():
        if kind == "linear":
            return state["layer"](state["x"])
        if "graph" in state:
            state["graph"].replay()
            return state["outs"]
        if kind in ("step", "layer"):
            return _step(state)
        if kind == "experts":
            return state["block"](state["x"], state["index"], state["weights"])
    w = state["w"]
    dense = nn.Linear(w.shape[1], w.shape[0], bias=False, device="meta").eval()
    dense.weight = nn.Parameter(w, requires_grad=False)
    model = optimize_model(nn.Sequential(dense), low_bit=state["low_bit"]).to("cuda")
    return model[0].weight.data


# ------------------------------------------------------------------ what a pass cannot do without

def _blob(case, n, k):
    qtype = ggml_tensor_qtype[case["qtype"]]
    return n * k // ggml.ggml_qk_size(qtype) * ggml.ggml_type_size(qtype)


def work(case):
    kind, size = case["kind"], 4 if case["dtype"] == "float32" else 2
    m = case.get("m", 0)
    if kind == "load":
        return {"bytes": case["n"] * case["k"] * 2 + _blob(case, case["n"], case["k"]), "flops": 0}
    if kind in ("linear", "train"):
        n, k = case["n"], case["k"]
        one = {"bytes": _blob(case, n, k) + m * (n + k) * size, "flops": 2 * m * n * k}
        return one if kind == "linear" else {"bytes": 2 * one["bytes"], "flops": 2 * one["flops"]}
    hidden, inter = case["hidden"], case["inter"]
    if kind == "experts":
        pairs = m * case["top_k"]
        return {"bytes": 3 * min(case["experts"], pairs) * _blob(case, inter, hidden) + 2 * m * hidden * size,
                "flops": 6 * pairs * inter * hidden}
    per_layer = [(hidden + 2 * case["kv"], hidden), (hidden, hidden), (2 * inter, hidden), (hidden, inter)]
    weights = case.get("layers", 1) * sum(n * k for n, k in per_layer)
    nbytes = case.get("layers", 1) * (sum(_blob(case, n, k) for n, k in per_layer) + m * (3 * hidden + 2 * case["kv"]) * size)
    vocab = case.get("vocab", 0)
    nbytes += 2 * m * hidden * size                    # the inputs, or embedded token and attention result
    if vocab:
        nbytes += _blob(case, vocab, hidden) + m * _blob(case, 1, hidden) + m * vocab * size
    return {"bytes": nbytes, "flops": 2 * m * (weights + vocab * hidden)}


def tolerance(case):
    if case["kind"] == "load":
        return "exact"
    # 16-bit results, and intermediate values or scaled weights rounded to 16 bits on the way; float32 activations
    # keep 16 mantissa bits or more
    return {"rel": {"float16": 2e-3, "bfloat16": 1e-2, "float32": 1e-5}[case["dtype"]]}
