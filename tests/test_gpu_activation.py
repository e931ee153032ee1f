"""SiLU and SwiGLU over their whole input range against the oracle, byte for byte: every bf16 input, binary32 inputs
over every exponent (where exp(-x) overflows, where x / d and 1 / d fall below the normal range), lengths that leave a
remainder past the last 16-byte vector and pointers that are not 16-byte aligned."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from attn_util import assert_bits_equal_nan_class as eq
from open_transformers_amd import _lib
from open_transformers_amd.nn import functional as F
from oracle import oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _inputs(bf16: bool) -> np.ndarray:
    if bf16:
        return (np.arange(65536, dtype=np.uint32) << 16).view(np.float32)
    rng = np.random.default_rng(4)
    u = rng.integers(0, 1 << 32, 200_000, dtype=np.uint64).astype(np.uint32).view(np.float32)
    near = np.concatenate([rng.uniform(-104.5, -80, 50_000), rng.uniform(-12, 12, 100_000)]).astype(np.float32)
    return np.concatenate([u, near, np.float32([0.0, -0.0, np.inf, -np.inf, np.nan, -88.72284, 88.72284, 1e-45])])


def _dev(a, bf16):
    return torch.from_numpy(np.ascontiguousarray(a)).to(torch.bfloat16 if bf16 else torch.float32).to(DEV)


@pytest.mark.parametrize("bf16", [True, False])
@pytest.mark.parametrize("offset,drop", [(0, 0), (1, 0), (0, 3)])
def test_silu_whole_range(bf16, offset, drop):
    print(f"silu bf16={bf16} offset={offset} drop={drop}", flush=True)
    x = _inputs(bf16)
    x = x[: x.size - drop]
    dy = np.random.default_rng(5).standard_normal(x.size).astype(np.float32)
    dy = _dev(dy, bf16).float().cpu().numpy()
    n = x.size
    bx, bd, by, bo = (torch.zeros(n + offset, dtype=torch.bfloat16 if bf16 else torch.float32, device=DEV)
                      for _ in range(4))
    bx[offset:] = _dev(x, bf16)
    bd[offset:] = _dev(dy, bf16)
    es, st = bx.element_size() * offset, torch.cuda.current_stream().cuda_stream
    lib, dt = _lib.load(), _lib.DTYPE_BF16 if bf16 else _lib.DTYPE_F32
    _lib.check(lib.otx_silu_fwd(bx.data_ptr() + es, by.data_ptr() + es, n, dt, st), "otx_silu_fwd")
    _lib.check(lib.otx_silu_bwd(bx.data_ptr() + es, bd.data_ptr() + es, bo.data_ptr() + es, n, dt, st), "otx_silu_bwd")
    torch.cuda.synchronize()
    eq(by[offset:].float().cpu().numpy(), orc.silu_fwd(x, out_bf16=bf16), "y")
    eq(bo[offset:].float().cpu().numpy(), orc.silu_bwd(x, dy, out_bf16=bf16), "dx")


@pytest.mark.parametrize("bf16", [True, False])
@pytest.mark.parametrize("cols", [8, 4096])
def test_swiglu_whole_range(bf16, cols):
    print(f"swiglu bf16={bf16} cols={cols}", flush=True)
    x = _inputs(bf16)
    x = x[: x.size // cols * cols].reshape(-1, cols)
    rng = np.random.default_rng(6)
    up, dh = (_dev(rng.standard_normal(x.shape).astype(np.float32), bf16).float().cpu().numpy() for _ in range(2))
    gu = _dev(np.concatenate([x, up], 1), bf16).requires_grad_()
    h = F.swiglu(gu)
    h.backward(_dev(dh, bf16))
    torch.cuda.synchronize()

    def rnd(a):
        return torch.from_numpy(a).to(torch.bfloat16).float().numpy() if bf16 else a

    with np.errstate(all="ignore"):
        y = orc.silu_fwd(x, out_bf16=bf16)
        eq(h.detach().float().cpu().numpy(), rnd(y * up), "h")
        want = np.concatenate([orc.silu_bwd(x, rnd(dh * up), out_bf16=bf16), rnd(dh * y)], 1)
    eq(gu.grad.float().cpu().numpy(), want, "dgu")
