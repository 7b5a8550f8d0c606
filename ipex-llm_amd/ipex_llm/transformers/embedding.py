"""Low-bit embedding table (reference: transformers/embedding.py:179-241).

The table is stored as a quantized blob; a lookup dequantizes only the rows it needs.
CPUEmbedding / DiskEmbedding of the reference keep the table off the accelerator and are not
part of the low-bit path built here.

The constructor's parameters are `torch.nn.Embedding`'s followed by `convert_shape_only` and `qtype`, in the
reference's order: `from_embedding` and the conversion pass hand them over by position."""
from typing import Optional

import torch
from torch import Tensor

from ipex_llm.transformers.native_ops import ops
from ipex_llm.utils.common import invalidInputError


class LowBitEmbedding(torch.nn.Embedding):
    def __init__(self, num_embeddings: int, embedding_dim: int, padding_idx: Optional[int] = None,
                 max_norm: Optional[float] = None, norm_type: float = 2., scale_grad_by_freq: bool = False,
                 sparse: bool = False, _weight: Optional[Tensor] = None, _freeze: bool = False, device=None,
                 dtype=None, convert_shape_only=None, qtype=None) -> None:
        from ipex_llm.transformers.low_bit_linear import FP4Params
        super().__init__(num_embeddings, embedding_dim, padding_idx, max_norm, norm_type, scale_grad_by_freq, sparse,
                         _weight, device=device, dtype=dtype)
        table = self.weight.data
        # the table lives on as a quantized parameter (quantized when the module reaches the GPU); `weight` shrinks
        # to an empty tensor that only records the model's dtype and device
        self.qweight = FP4Params(table, requires_grad=False, quantized=False, _shape=None,
                                 convert_shape_only=convert_shape_only, qtype=qtype, in_features=embedding_dim)
        self.weight = torch.nn.Parameter(torch.empty(0, 0, dtype=table.dtype, device=table.device), requires_grad=False)

    def forward(self, x: Tensor):
        from ipex_llm.transformers.low_bit_linear import dequantize_rows
        table = self.qweight
        if table.quantized and table._shape is not None:
            # one native call: the rows come out in the model's dtype (None: not the plain case, the steps below)
            rows = ops.embedding(x, table, table.qtype, self.num_embeddings, self.embedding_dim, self.weight)
            if rows is not None:
                return rows
        invalidInputError(x.device.type == "cuda", "`LowBitEmbedding` only supports GPU now.")
        invalidInputError(self.qweight.quantized and self.qweight.device == x.device,
                          "move the module to the GPU first: the table is quantized on the way")
        result = dequantize_rows(x.contiguous(), self.qweight.data, self.qweight.qtype,
                                 self.embedding_dim, self.num_embeddings, layout=self.qweight.blob_layout)
        return result.to(self.weight.dtype)

    @classmethod
    def from_embedding(cls, embedding: torch.nn.Embedding, convert_shape_only, qtype):
        e = embedding
        return cls(e.num_embeddings, e.embedding_dim, e.padding_idx, e.max_norm, e.norm_type, e.scale_grad_by_freq,
                   e.sparse, e.weight.data, True, e.weight.device, e.weight.dtype, convert_shape_only, qtype)
