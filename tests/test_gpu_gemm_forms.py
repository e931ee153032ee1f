"""The GEMM forms (the small ones on v_mfma_f32_16x16x4_f32: four serial fmas per instruction) against the serial-fold
oracle where they can go wrong: every remainder of R by the stage length of the small forms (64 and 128), one to more
stages than the LDS slots, both operand layouts of each side, padded row pitches, and operands whose fold order and
rounding show in every output (cancellations over 2^24, subnormals, signed zeros, infinities)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from attn_util import assert_bits_equal_nan_class as eq
from open_transformers_amd import synthetic
from open_transformers_amd.nn import functional as F
from oracle import oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
M, N = 128, 256  # two wide tiles: the library takes the 32 x 32 form


def _operand(rng, rows, R, kind):
    x = rng.standard_normal((rows, R))
    if kind == "cancel":
        x = x * 2.0 ** rng.integers(-12, 13, (rows, R))
    elif kind == "tiny":
        x = x * 2.0 ** rng.integers(-75, -55, (rows, R))
        x[rng.random((rows, R)) < 0.1] = -0.0
        x[rng.random((rows, R)) < 0.1] = 1e-39
    elif kind == "inf":
        x[1, R // 2], x[rows - 1, 3] = np.inf, -np.inf
    return synthetic.round_to_bf16(x.astype(np.float32))


def _dev(a, r_contiguous, pad):
    """(tensor, row stride, r stride) of a [rows, R] operand in either layout, rows padded by ``pad`` elements."""
    a = a if r_contiguous else np.ascontiguousarray(a.T)
    buf = torch.zeros(a.shape[0], a.shape[1] + pad, dtype=torch.bfloat16, device=DEV)
    buf[:, :a.shape[1]] = torch.from_numpy(a).to(torch.bfloat16).to(DEV)
    ld = a.shape[1] + pad
    return (buf, (ld, 1)) if r_contiguous else (buf, (1, ld))


@pytest.mark.parametrize("R", [32, 64, 96, 128, 160, 224, 352, 512, 544, 1120])
@pytest.mark.parametrize("kind", ["cancel", "tiny", "inf"])
def test_small_forms_match_the_serial_fold(R, kind):
    print(f"gemm forms R{R} {kind}", flush=True)
    rng = np.random.default_rng(R)
    a, b = _operand(rng, M, R, kind), _operand(rng, N, R, kind)
    with np.errstate(all="ignore"):
        ref, ref32 = orc.gemm(a, b), orc.gemm(a, b, out_bf16=False)
    for arc in (True, False):
        for brc in (True, False):
            ta, sa = _dev(a, arc, 8)
            tb, sb = _dev(b, brc, 16)
            for variant in range(5):
                y = F.gemm_bf16(ta, sa, tb, sb, M, N, R, variant=variant)
                y32 = F.gemm_bf16(ta, sa, tb, sb, M, N, R, out_dtype=torch.float32, variant=variant)
                torch.cuda.synchronize()
                eq(y.float().cpu().numpy(), ref, f"bf16 result, layouts {arc} {brc}, variant {variant}")
                eq(y32.cpu().numpy(), ref32, f"binary32 result, layouts {arc} {brc}, variant {variant}")


@pytest.mark.parametrize("shape", [(128, 256, 512), (1024, 1024, 96), (1280, 5632, 64), (2048, 4096, 64)])
def test_every_form_gives_the_chosen_ones_bytes(shape):
    """Products of few to many tiles (the library's choice goes from 32 x 32 to the wide tiles), every forced form and
    layout against the choice."""
    m, n, r = shape
    print(f"gemm forms {shape}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(m + n)
    a, b = (torch.randn(rows, r, device=DEV, generator=g).bfloat16() for rows in (m, n))
    ref = F.gemm_bf16(a, (r, 1), b, (r, 1), m, n, r)
    at, bt = a.t().contiguous(), b.t().contiguous()
    for ta, sa in ((a, (r, 1)), (at, (1, m))):
        for tb, sb in ((b, (r, 1)), (bt, (1, n))):
            for variant in range(5):
                y = F.gemm_bf16(ta, sa, tb, sb, m, n, r, variant=variant)
                assert torch.equal(y.view(torch.int16), ref.view(torch.int16)), (sa, sb, variant)
