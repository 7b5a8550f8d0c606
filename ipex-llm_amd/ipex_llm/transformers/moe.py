"""Mixture-of-experts feed-forward on low-bit experts.

The reference has no fused path for a Mixtral-style block at prefill: the Hugging Face block
loops over the experts and calls each expert's (converted) LowBitLinear on the rows routed to
it, then index_adds the weighted result (the same pattern as the reference's own
transformers/models/qwen2_moe.py:375-430).  `moe_ffn_reference` is that loop; `moe_ffn_grouped` and
`LowBitExperts` compute the same thing in one native call (csrc/moe.hip): the (token, expert) pairs sorted by
expert, the fused gate/up projection with the activation in its epilogue, the down projection and the weighted
sum - or, while there are no more pairs than experts, two launches of the streaming kernel.  What that call does
not take runs as torch operators around the two grouped launches (`_grouped_steps`).
"""
import array

import torch
import torch.nn as nn
import torch.nn.functional as F

import ipex_llm.ggml.model.llama.llama_cpp as ggml
from ipex_llm.transformers.low_bit_linear import _DT, _as_u8, _stream
from ipex_llm.transformers.native_ops import ops
from ipex_llm.utils.common import invalidInputError


def route_top_k(router_logits: torch.Tensor, top_k: int = 2):
    """softmax over experts in fp32, top-k, renormalised (Hugging Face Mixtral semantics)."""
    probs = F.softmax(router_logits.float(), dim=-1)
    weights, experts = torch.topk(probs, top_k, dim=-1)
    weights = weights / weights.sum(dim=-1, keepdim=True)
    return weights, experts


class ExpertWeights:
    """Device pointers of one projection of every expert ([N, K] tiled blobs of one qtype)."""

    def __init__(self, linears):
        invalidInputError(len(linears) > 0, "no experts")
        l0 = linears[0]
        self.qtype, self.out_len, self.in_len = l0.qtype, l0.out_len, l0.in_len
        for lin in linears:
            invalidInputError(lin.weight.device.type == "cuda" and lin.weight.quantized
                              and (lin.qtype, lin.out_len, lin.in_len) == (self.qtype, self.out_len, self.in_len),
                              "experts must be quantized, on the GPU and of one shape / qtype")
        invalidInputError(ggml.lowbit_tileable(self.qtype, self.out_len, self.in_len),
                          "grouped experts need out_features % 16 == 0 and in_features % 128 == 0")
        want = ggml.lowbit_blob_bytes(self.qtype, self.out_len * self.in_len)
        for lin in linears:
            invalidInputError(lin.weight.data.device == l0.weight.data.device
                              and lin.weight.blob_layout == ggml.LAYOUT_TILED
                              and _as_u8(lin.weight.data).numel() == want and lin.weight.data.is_contiguous(),
                              "every expert must hold a tiled blob of the common shape on one GPU")
        self.linears = list(linears)
        self.blobs = [_as_u8(lin.weight.data) for lin in linears]        # keeps the storage alive
        addresses = array.array("Q", [b.data_ptr() for b in self.blobs])
        self.ptrs = torch.tensor(addresses.tolist(), dtype=torch.int64, device=l0.weight.device)
        self.held = (tuple(lin._parameters for lin in linears), addresses.tobytes())      # what `holds` compares
        self.shape = (self.out_len, self.in_len, len(self.blobs))

    def holds(self, device):
        """Whether every layer still has the weight that the pointer table, a snapshot, points to."""
        return self.ptrs.device == device and ops.holds(*self.held)

    def check(self, device):
        """Refuses to launch if a layer was moved or re-quantized since the table was built."""
        invalidInputError(self.holds(device),
                          "an expert weight was moved or replaced after ExpertWeights was built; build it again")


def _check_grouped(x_sorted, group_offsets, experts):
    invalidInputError(x_sorted.dim() == 2 and x_sorted.shape[1] == experts.in_len and x_sorted.dtype in _DT
                      and x_sorted.dtype != torch.float32, "x must be [rows, K] in fp16 / bf16")
    invalidInputError(group_offsets.dtype == torch.int32 and group_offsets.numel() == len(experts.blobs) + 1
                      and group_offsets.device == x_sorted.device, "group_offsets must be int32 [E + 1] on the GPU")
    experts.check(x_sorted.device)


def grouped_forward(x_sorted: torch.Tensor, group_offsets: torch.Tensor, experts: ExpertWeights):
    """y[r] = x_sorted[r] @ dequant(W[e])^T for group_offsets[e] <= r < group_offsets[e+1]."""
    _check_grouped(x_sorted, group_offsets, experts)
    x_sorted = x_sorted.contiguous()
    rows = x_sorted.shape[0]
    y = torch.empty((rows, experts.out_len), dtype=x_sorted.dtype, device=x_sorted.device)
    if rows:
        n_exp = len(experts.blobs)
        ws_bytes = ggml.lowbit_grouped_workspace_bytes(n_exp, rows, experts.out_len, experts.in_len)
        ws = torch.empty(max(ws_bytes, 16), dtype=torch.uint8, device=x_sorted.device)
        with torch.cuda.device(x_sorted.device):
            ggml.lowbit_grouped_forward_ws(x_sorted.data_ptr(), experts.ptrs.data_ptr(), y.data_ptr(),
                                           group_offsets.data_ptr(), n_exp, rows, experts.qtype, _DT[x_sorted.dtype],
                                           experts.out_len, experts.in_len, ws.data_ptr(), ws_bytes, _stream())
    return y


def grouped_mlp_forward(x_sorted: torch.Tensor, group_offsets: torch.Tensor, gates: ExpertWeights,
                        ups: ExpertWeights, act: int = 0):
    """h[r] = act(x_sorted[r] @ Wg[e]^T) * (x_sorted[r] @ Wu[e]^T) for the rows of group e, in one launch
    (act: 0 = SiLU, 1 = tanh-GELU, as in mlp_forward_xpu)."""
    _check_grouped(x_sorted, group_offsets, gates)
    invalidInputError((ups.qtype, ups.out_len, ups.in_len) == (gates.qtype, gates.out_len, gates.in_len)
                      and len(ups.blobs) == len(gates.blobs), "gate and up experts do not fit together")
    ups.check(x_sorted.device)
    x_sorted = x_sorted.contiguous()
    rows = x_sorted.shape[0]
    h = torch.empty((rows, gates.out_len), dtype=x_sorted.dtype, device=x_sorted.device)
    if rows:
        with torch.cuda.device(x_sorted.device):
            ggml.lowbit_grouped_mlp_forward(x_sorted.data_ptr(), gates.ptrs.data_ptr(), ups.ptrs.data_ptr(),
                                            h.data_ptr(), group_offsets.data_ptr(), len(gates.blobs), rows,
                                            gates.qtype, _DT[x_sorted.dtype], gates.out_len, gates.in_len, act,
                                            _stream())
    return h


def moe_forward_vec(x: torch.Tensor, topk_ids: torch.Tensor, topk_weight: torch.Tensor, gates: ExpertWeights,
                    ups: ExpertWeights, downs: ExpertWeights, act: int = 0):
    """xe_linear.moe_forward_vec (models/deepseek.py:290-315 of the reference): one token through its top-k
    experts in two launches.  Nothing is read back to the host: the expert ids stay on the GPU.
    x [1, hidden]; topk_ids / topk_weight [1, top_k]; returns [1, hidden]."""
    hidden, inter = gates.in_len, gates.out_len
    invalidInputError(x.dim() == 2 and x.shape == (1, hidden) and x.dtype in (torch.float16, torch.bfloat16),
                      "moe_forward_vec expects one fp16 / bf16 row of x")
    invalidInputError((ups.qtype, ups.out_len, ups.in_len) == (gates.qtype, inter, hidden)
                      and (downs.qtype, downs.out_len, downs.in_len) == (gates.qtype, hidden, inter),
                      "gate / up / down experts do not fit together")
    for table in (gates, ups, downs):
        table.check(x.device)
    top_k = topk_ids.numel()
    invalidInputError(topk_weight.numel() >= top_k, "every expert id needs a weight")
    ids = topk_ids.reshape(-1).to(x.device, torch.int32)
    rw = topk_weight.reshape(-1).to(x.device, torch.float32)
    xc = x.contiguous()
    work = torch.empty((top_k, inter), dtype=x.dtype, device=x.device)
    y = torch.empty((1, hidden), dtype=x.dtype, device=x.device)
    with torch.cuda.device(x.device):
        ggml.lowbit_moe_forward(xc.data_ptr(), ids.data_ptr(), rw.data_ptr(), top_k, len(gates.blobs),
                                gates.ptrs.data_ptr(), ups.ptrs.data_ptr(), downs.ptrs.data_ptr(), work.data_ptr(),
                                y.data_ptr(), gates.qtype, _DT[x.dtype], hidden, inter, act, _stream())
    return y


def moe_ffn_reference(hidden, router_logits, w1, w3, w2, top_k=2):
    """The per-expert loop: w1/w3/w2 are lists of LowBitLinear (gate, up, down)."""
    weights, experts = route_top_k(router_logits, top_k)
    out = torch.zeros_like(hidden)
    for e in range(len(w1)):
        tok, slot = torch.where(experts == e)
        if tok.numel() == 0:
            continue
        xe = hidden[tok]
        he = F.silu(w1[e](xe)) * w3[e](xe)
        ye = w2[e](he) * weights[tok, slot].unsqueeze(-1).to(hidden.dtype)
        out.index_add_(0, tok, ye.to(hidden.dtype))
    return out


def _native(hidden, index, weights, gates: ExpertWeights, ups: ExpertWeights, downs: ExpertWeights, act):
    """The block in one native call (csrc/moe.hip), None for what that does not take; refuses tables that do not fit
    together."""
    inter, width, n_exp = gates.shape
    invalidInputError(ups.qtype == gates.qtype and ups.shape == gates.shape and downs.shape == (width, inter, n_exp),
                      "gate / up / down experts do not fit together")
    if downs.qtype != gates.qtype:                       # the call decodes all three in one format
        return None
    return ops.experts(hidden, index, weights, gates.ptrs, ups.ptrs, downs.ptrs, gates.qtype, width, inter, act)


def _grouped_steps(hidden, index, weights, gates: ExpertWeights, ups: ExpertWeights, downs: ExpertWeights, act):
    """The experts' weighted sum as torch operators around the two grouped launches, for what the native call does not
    take: routing weights that want a gradient, down weights of another format than the gate's, no tokens, more than 64
    experts per token or 4096 in all, indices or weights on another device.  A pair whose index names no expert counts nothing."""
    top_k, n_exp = index.shape[1], len(gates.blobs)
    invalidInputError(index.shape[0] <= hidden.shape[0] and weights.numel() == index.numel(),
                      "every row of the indices needs a row of hidden, every index a weight")
    expert = index.reshape(-1).to(hidden.device, torch.int64)
    none = (expert < 0) | (expert >= n_exp)
    expert, order = torch.sort(expert.masked_fill(none, n_exp), stable=True)
    offsets = torch.searchsorted(expert, torch.arange(n_exp + 1, device=hidden.device), out_int32=True)
    tok = torch.div(order, top_k, rounding_mode="floor")
    h = grouped_mlp_forward(hidden[tok], offsets, gates, ups, act)
    none = none[order].unsqueeze(-1)
    w = weights.reshape(-1).to(hidden.device)[order].unsqueeze(-1).to(hidden.dtype).masked_fill(none, 0)
    y = grouped_forward(h, offsets, downs).masked_fill(none, 0) * w
    out = torch.zeros_like(hidden)
    out.index_add_(0, tok, y)
    return out


def moe_ffn_grouped(hidden, router_logits, g1: ExpertWeights, g3: ExpertWeights, g2: ExpertWeights, top_k=2):
    """Same result in one call of the experts block (csrc/moe.hip)."""
    weights, experts = route_top_k(router_logits, top_k)
    for table in (g1, g3, g2):
        table.check(hidden.device)
    out = _native(hidden, experts, weights, g1, g3, g2, 0)
    return _grouped_steps(hidden, experts, weights, g1, g3, g2, 0) if out is None else out


def activation_code(act_fn):
    """0 (SiLU) / 1 (tanh-GELU) for the activations the fused kernels know, None for any other."""
    name = act_fn.__class__.__name__
    if isinstance(act_fn, nn.SiLU) or name in ("SiLUActivation", "SiLU"):
        return 0
    if (isinstance(act_fn, nn.GELU) and act_fn.approximate == "tanh") or name in ("PytorchGELUTanh", "GELUTanh",
                                                                               "NewGELUActivation"):
        return 1
    return None


class LowBitExperts(nn.Module):
    """The experts of a sparse mixture-of-experts block with low-bit weights.

    With the transformers version the reference pins (4.37) every expert is a small module of three nn.Linear
    layers, which its `_replace_with_low_bit_linear` turns into LowBitLinear one by one (convert.py:469-748) and
    the block's Python loop calls in turn.  Current transformers keep all experts of a block in one module with two
    3-D parameters, `gate_up_proj` [E, 2 I, H] and `down_proj` [E, H, I], and the call
    `experts(hidden_states [T, H], top_k_index [T, k], top_k_weights [T, k]) -> [T, H]` (MixtralExperts and its
    siblings).  This module takes that one's place: each expert's three weights become LowBitLinear layers
    (`gate[e]`, `up[e]`, `down[e]`, so that save_low_bit / load_low_bit carry them like any other), and on the GPU the
    call is one native call (see the head of this file).  With anything else - host tensors, float32 activations,
    training, an activation the kernels do not know, shapes without a tiled layout - it is the per-expert loop over the
    LowBitLinear layers."""

    def __init__(self, num_experts, hidden_dim, intermediate_dim, qtype, act_fn, enable_scale_search=False):
        super().__init__()
        from ipex_llm.transformers.low_bit_linear import LowBitLinear
        self.num_experts, self.hidden_dim, self.intermediate_dim, self.qtype = num_experts, hidden_dim, intermediate_dim, qtype
        self.act_fn = act_fn

        def layers(in_f, out_f):
            return nn.ModuleList([LowBitLinear(in_f, out_f, qtype, bias=False, enable_scale_search=enable_scale_search)
                                  for _ in range(num_experts)])
        self.gate, self.up = layers(hidden_dim, intermediate_dim), layers(hidden_dim, intermediate_dim)
        self.down = layers(intermediate_dim, hidden_dim)
        self.__dict__["_tables"] = None

    @classmethod
    def from_fused(cls, module, qtype, convert_shape_only=False, enable_scale_search=False):
        """From a module that holds `gate_up_proj` [E, 2 I, H], `down_proj` [E, H, I] and `act_fn`."""
        from ipex_llm.transformers.low_bit_linear import FP4Params
        gate_up, down = module.gate_up_proj.data, module.down_proj.data
        n_exp, two_i, hidden = gate_up.shape
        inter = two_i // 2
        invalidInputError(tuple(down.shape) == (n_exp, hidden, inter), "gate_up_proj / down_proj shapes do not fit together")
        new = cls(n_exp, hidden, inter, qtype, module.act_fn, enable_scale_search)
        device = gate_up.device

        def param(w, in_features):
            return FP4Params(data=w.contiguous() if w.device.type != "meta" else w, requires_grad=False, quantized=False,
                             _shape=None, convert_shape_only=convert_shape_only, qtype=qtype, in_features=in_features,
                             enable_scale_search=enable_scale_search).to(device)
        for e in range(n_exp):
            new.gate[e]._parameters["weight"] = param(gate_up[e, :inter], hidden)
            new.up[e]._parameters["weight"] = param(gate_up[e, inter:], hidden)
            new.down[e]._parameters["weight"] = param(down[e], inter)
        if not module.training:
            new.eval()
        new.requires_grad_(False)
        return new

    def _expert_tables(self, x):
        """Pointer tables of the three projections, built on first use and again when a weight has moved; None where the
        call is not one for the grouped kernels."""
        if not x.is_cuda or x.dtype not in (torch.float16, torch.bfloat16) or self.training \
                or activation_code(self.act_fn) is None:
            return None
        tables = self.__dict__["_tables"]
        if tables is None or not all(t.holds(x.device) for t in tables):
            self.__dict__["_tables"] = None
            w = self.gate[0].weight
            if not (w.quantized and w.data.device == x.device
                    and ggml.lowbit_tileable(self.qtype, self.intermediate_dim, self.hidden_dim)
                    and ggml.lowbit_tileable(self.qtype, self.hidden_dim, self.intermediate_dim)):
                return None
            tables = tuple(ExpertWeights(list(layers)) for layers in (self.gate, self.up, self.down))
            self.__dict__["_tables"] = tables
        return tables

    def forward(self, hidden_states, top_k_index, top_k_weights):
        if top_k_index.shape[0] == 0:
            return torch.zeros_like(hidden_states)
        tables = self._expert_tables(hidden_states)
        if tables is None:
            return self._loop(hidden_states, top_k_index, top_k_weights)
        act = activation_code(self.act_fn)
        y = _native(hidden_states, top_k_index, top_k_weights, *tables, act)
        if y is None and top_k_index.shape[0] == 1 and top_k_index.shape[1] <= 64:
            return moe_forward_vec(hidden_states, top_k_index, top_k_weights, *tables, act)
        return _grouped_steps(hidden_states, top_k_index, top_k_weights, *tables, act) if y is None else y

    def _loop(self, hidden_states, top_k_index, top_k_weights):
        out = torch.zeros_like(hidden_states)
        for e in range(self.num_experts):
            tok, slot = torch.where(top_k_index == e)
            if tok.numel() == 0:
                continue
            xe = hidden_states[tok]
            he = self.down[e](self.act_fn(self.gate[e](xe)) * self.up[e](xe))
            out.index_add_(0, tok, (he * top_k_weights[tok, slot, None]).to(out.dtype))
        return out
