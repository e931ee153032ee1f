"""ROCm operators for the decoder layer around the attention.

Mirrors the repop operators the reference's modules call:
  linear(x, w)          repop.nn.linear.Linear forward (src/pretrain/model/modules/_linear.py:31-65)
  rms_norm(x, w, eps)   repop.nn.rmsnorm.rms_norm (src/pretrain/model/modules/norm_repop.py:19-22)
  silu(x)               repop.nn.activations.silu (src/pretrain/model/modules/ffn_repop.py:28-36)
and the torch compositions around them, each fused into one pass:
  swiglu(gu)            gate, up = gu.chunk(2, -1); silu(gate) * up (ffn_repop.py:52-54)
  rope_heads(x, c, s)   apply_rope(x, c, s).transpose(1, 2).contiguous()
                        (rope.py:103-125, attention_repop.py:143-149)
  heads(x)              x.transpose(1, 2).contiguous() (attention_repop.py:150)
  merge_heads(o)        o.transpose(1, 2).contiguous().view(B, T, H * D) (attention_repop.py:155)
Each is an autograd node of csrc/otx_autograd.cpp over the C ABI of libotx_attn.so: bf16 in,
binary32 arithmetic in a fixed order, bf16 out, and for the compositions the
bytes torch's own forward and autograd backward give; weight gradients come
back in the weight's dtype.  GPU tensors only; there is no CPU fallback.
"""

from __future__ import annotations

import torch

from .. import _lib
from . import _nodes

__all__ = ["linear", "rms_norm", "silu", "swiglu", "rope_heads", "heads", "merge_heads"]

_DT = {torch.bfloat16: _lib.DTYPE_BF16, torch.float32: _lib.DTYPE_F32}


def _stream(t: torch.Tensor) -> int:
    return torch.cuda.current_stream(t.device).cuda_stream


def _need_gpu(*ts: torch.Tensor) -> None:
    for t in ts:
        if t.device.type != "cuda":
            raise RuntimeError(f"tensor on {t.device}: this operator is the ROCm (HIP) backend and only accepts GPU tensors")


def gemm_bf16(a: torch.Tensor, a_strides: tuple[int, int], b: torch.Tensor, b_strides: tuple[int, int],
              M: int, N: int, R: int, out_dtype: torch.dtype = torch.bfloat16, variant: int = 0) -> torch.Tensor:
    """C[M, N] with C[i][j] = serial fold over r of A(i, r) * B(j, r) (strides in elements).
    ``variant``: 0 lets the library choose the tile form, 1, 2, 3 and 4 force the wide
    (128 x 128), the narrow (128 x 64, where both operands' first stride is 1), and the
    small ones (64 x 64 and 32 x 32); same bytes."""
    if a.dtype != torch.bfloat16 or b.dtype != torch.bfloat16:
        raise ValueError("gemm_bf16 takes bfloat16 operands")
    c = torch.empty((M, N), dtype=out_dtype, device=a.device)
    lib = _lib.load()
    rc = lib.otx_gemm_bf16_ex(a.data_ptr(), a_strides[0], a_strides[1], b.data_ptr(), b_strides[0], b_strides[1],
                              c.data_ptr(), N, M, N, R, _DT[out_dtype], variant, _stream(a))
    _lib.check(rc, "otx_gemm_bf16_ex")
    return c


def linear(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """y = x @ w^T (no bias), bf16 operands, serial binary32 fold, bf16 result."""
    _need_gpu(x, w)
    return _nodes.call("linear", x, w)


def rms_norm(x: torch.Tensor, w: torch.Tensor, eps: float) -> torch.Tensor:
    """RMSNorm over the last dimension; output in x's dtype, rstd kept for backward."""
    _need_gpu(x, w)
    if x.dtype not in _DT:
        raise ValueError(f"dtype {x.dtype} not supported")
    return _nodes.call("rms_norm", x, w, float(eps))


def silu(x: torch.Tensor) -> torch.Tensor:
    """SiLU with a correctly rounded exp, in x's dtype."""
    _need_gpu(x)
    if x.dtype not in _DT:
        raise ValueError(f"dtype {x.dtype} not supported")
    return _nodes.call("silu", x)


def swiglu(gu: torch.Tensor) -> torch.Tensor:
    """silu(gate) * up for gate, up = gu.chunk(2, -1), in one pass; the last
    dimension of gu is 2F with F a multiple of 8."""
    _need_gpu(gu)
    if gu.dtype not in _DT:
        raise ValueError(f"dtype {gu.dtype} not supported")
    if gu.shape[-1] % 16:
        raise ValueError(f"swiglu: last dimension {gu.shape[-1]} is not a multiple of 16")
    return _nodes.call("swiglu", gu)


def rope_heads(x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor) -> torch.Tensor:
    """RoPE of x [B, T, H, D] (interleaved pairs, cos/sin binary32 [T, D/2]) into
    the attention layout [B, H, T, D]."""
    _need_gpu(x, cos, sin)
    if x.dtype not in _DT:
        raise ValueError(f"dtype {x.dtype} not supported")
    if x.dim() != 4 or x.shape[-1] % 8:
        raise ValueError(f"rope_heads takes x [B, T, H, D] with D a multiple of 8, got {tuple(x.shape)}")
    T, D = x.shape[1], x.shape[3]
    for name, t in (("cos", cos), ("sin", sin)):
        if t.dtype != torch.float32 or tuple(t.shape) != (T, D // 2):
            raise ValueError(f"rope_heads: {name} must be binary32 [{T}, {D // 2}], got {t.dtype} {tuple(t.shape)}")
    return _nodes.call("rope_heads", x, cos.contiguous(), sin.contiguous())


def heads(x: torch.Tensor) -> torch.Tensor:
    """[B, T, H, D] -> [B, H, T, D] (contiguous)."""
    _need_gpu(x)
    if x.dtype not in _DT or x.dim() != 4 or x.shape[-1] % 8:
        raise ValueError(f"heads takes a bf16/binary32 [B, T, H, D] tensor with D a multiple of 8, got {x.dtype} "
                         f"{tuple(x.shape)}")
    return _nodes.call("swap_heads", x)


def merge_heads(o: torch.Tensor) -> torch.Tensor:
    """[B, H, T, D] -> [B, T, H * D] (contiguous)."""
    _need_gpu(o)
    if o.dtype not in _DT or o.dim() != 4 or o.shape[-1] % 8:
        raise ValueError(f"merge_heads takes a bf16/binary32 [B, H, T, D] tensor with D a multiple of 8, got "
                         f"{o.dtype} {tuple(o.shape)}")
    B, H, T, D = o.shape
    return _nodes.call("swap_heads", o).view(B, T, H * D)
