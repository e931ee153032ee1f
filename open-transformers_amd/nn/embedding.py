"""ROCm implementation of ``repop.nn.embedding.Embedding``.

The reference's untied embedding (src/pretrain/model/modules/
embedding_repop.py:33-40) looks tokens up with repop's Embedding, a drop-in
for ``torch.nn.Embedding`` whose backward is a deterministic fixed-order
scatter-add (docs/MODEL_OP_DTYPE_TRACE.md:75,106).  Here the forward is a row
gather and the backward folds, per token id, the gradient rows of its
positions in ascending position order in binary32, on the gfx950 kernels of
csrc/embedding.hip.
"""

from __future__ import annotations

import torch
import torch.nn as nn

from . import _nodes

__all__ = ["Embedding", "embedding"]

_DTYPES = (torch.bfloat16, torch.float32)


def embedding(ids: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """Rows ``weight[ids]``; the backward folds each id's gradient rows in position order."""
    if weight.device.type != "cuda":
        raise RuntimeError(f"weight is on {weight.device}: this Embedding is the ROCm (HIP) backend")
    if weight.dtype not in _DTYPES or weight.dim() != 2 or not weight.is_contiguous():
        raise ValueError("weight must be a contiguous 2-D bfloat16 or float32 tensor")
    if ids.device != weight.device:
        # the kernels dereference the ids pointer on the GPU: a host pointer would fault.
        # RuntimeError, as torch.nn.Embedding raises for the same mismatch.
        raise RuntimeError(f"ids are on {ids.device} but weight is on {weight.device}: "
                           "Expected all tensors to be on the same device")
    return _nodes.call("embedding", ids, weight)


class Embedding(nn.Module):
    """``Embedding(num_embeddings, embedding_dim)`` with ``.weight`` [V, D]."""

    def __init__(self, num_embeddings: int, embedding_dim: int, dtype=torch.bfloat16, device=None):
        super().__init__()
        self.num_embeddings, self.embedding_dim = num_embeddings, embedding_dim
        self.weight = nn.Parameter(torch.empty(num_embeddings, embedding_dim, dtype=dtype, device=device))

    def forward(self, ids: torch.Tensor) -> torch.Tensor:
        return embedding(ids, self.weight)
