"""GPU parity of the fused cross-entropy + z-loss (csrc/loss.hip) against the
CPU oracle, byte for byte: the per-row statistics (max, Z, lse, d, q), the two
scalars and the logit gradient.

Shapes follow the reference's own tests of the fused loss
(tests/test_fused_loss.py: N 48 x V 512 binary32, N 40 x V 320 bf16, both
coefficients) plus ragged and unaligned vocabularies, single rows and columns,
labels at both ends, a label outside the vocabulary, and the OPEN-1B lm-head
shape (V = 128256, configs/model/llama3_1b_proxy_repop.yaml) with all rows'
statistics and a slice of rows' gradients checked.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from attn_util import assert_bits_equal
from oracle import oracle as orc
from open_transformers_amd import synthetic
from open_transformers_amd.nn import loss as L

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _inputs(N, V, dtype, seed, scale=1.0):
    rng = np.random.default_rng(seed)
    x = (rng.standard_normal((N, V)) * scale).astype(np.float32)
    if dtype == "bf16":
        x = synthetic.round_to_bf16(x)
    lab = rng.integers(0, V, N).astype(np.int64)
    lab[0] = 0
    lab[-1] = V - 1
    return x, lab


def _gpu(x, dtype):
    return torch.from_numpy(x).to(torch.bfloat16 if dtype == "bf16" else torch.float32).to(DEV)


CASES = [
    pytest.param(48, 512, "f32", 1e-4, id="ref-shape-f32"),
    pytest.param(48, 512, "f32", 0.0, id="ref-shape-f32-coeff0"),
    pytest.param(40, 320, "bf16", 1e-4, id="ref-shape-bf16"),
    pytest.param(40, 320, "bf16", 0.0, id="ref-shape-bf16-coeff0"),
    pytest.param(33, 1000, "bf16", 1e-5, id="ragged-vocab"),
    pytest.param(17, 1001, "bf16", 1e-4, id="unaligned-vocab"),
    pytest.param(9, 999, "f32", 1e-4, id="unaligned-f32"),
    pytest.param(1, 7, "bf16", 1e-4, id="one-row"),
    pytest.param(64, 1, "bf16", 1e-4, id="one-column"),
    pytest.param(300, 4096, "bf16", 1e-4, id="many-rows"),
]


@pytest.mark.parametrize("N,V,dtype,coeff", CASES)
def test_loss_fwd_bwd_bitexact(N, V, dtype, coeff):
    print(f"loss case N={N} V={V} {dtype} coeff={coeff}", flush=True)
    x, lab = _inputs(N, V, dtype, seed=N + V, scale=3.0)
    ce_r, z_r, st_r = orc.ce_zloss_fwd(x, lab, coeff)
    logits = _gpu(x, dtype).requires_grad_()
    labels = torch.from_numpy(lab).to(DEV)
    ce, z = L.fused_ce_z_loss(logits, labels, coeff)
    (2.0 * ce + 3.0 * z).backward()
    torch.cuda.synchronize()
    _, _, st = L.ce_zloss_forward(logits.detach(), labels, coeff)
    assert_bits_equal(st.cpu().numpy(), st_r, "row statistics")
    assert_bits_equal(np.array([ce.item(), z.item()], np.float32), np.array([ce_r, z_r], np.float32), "ce, z")
    g_r = orc.ce_zloss_bwd(x, lab, st_r, coeff, gce=2.0, gz=3.0, out_bf16=dtype == "bf16")
    assert_bits_equal(logits.grad.float().cpu().numpy(), g_r, "logit gradient")


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_loss_wide_logit_spread(dtype):
    """Logits N(0, 40^2): most probabilities exp(x - m) / Z fall below the normal
    range or to zero, where the backward's quotient takes the exact division
    instead of the binary64 reciprocal; both paths against the oracle."""
    N, V = 64, 2048
    print(f"loss wide spread {dtype}", flush=True)
    x, lab = _inputs(N, V, dtype, seed=11, scale=40.0)
    ce_r, z_r, st_r = orc.ce_zloss_fwd(x, lab, 1e-4)
    logits = _gpu(x, dtype).requires_grad_()
    ce, z = L.fused_ce_z_loss(logits, torch.from_numpy(lab).to(DEV), 1e-4)
    (ce + z).backward()
    torch.cuda.synchronize()
    g_r = orc.ce_zloss_bwd(x, lab, st_r, 1e-4, out_bf16=dtype == "bf16")
    sub = np.count_nonzero((np.abs(g_r) < np.float32(2.0 ** -126)) & (g_r != 0))
    assert sub > 0, "the case must reach gradients below the normal range"
    assert_bits_equal(logits.grad.float().cpu().numpy(), g_r, "logit gradient")


def test_bad_label_gives_nan():
    x, lab = _inputs(8, 64, "bf16", seed=5)
    lab[3] = 64
    ce, _ = L.fused_ce_z_loss(_gpu(x, "bf16"), torch.from_numpy(lab).to(DEV), 1e-4)
    assert np.isnan(ce.item())


def test_open1b_lm_head_shape():
    """N = 4 x 2048 rows of the 128256-token vocabulary (bf16 logits, coeff 1e-4):
    every row's statistics and both scalars against the oracle, and the gradient
    of 64 rows (the backward is row-independent given the 1/N scale)."""
    N, V = 8192, 128256
    print(f"loss OPEN-1B lm-head N={N} V={V}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(77)
    logits = (torch.randn(N, V, device=DEV, generator=gen) * 2.0).to(torch.bfloat16).requires_grad_()
    labels = torch.randint(0, V, (N,), device=DEV, generator=gen)
    x = logits.detach().float().cpu().numpy()
    lab = labels.cpu().numpy()
    ce, z = L.fused_ce_z_loss(logits, labels, 1e-4)
    (ce + z).backward()
    torch.cuda.synchronize()
    ce_r, z_r, st_r = orc.ce_zloss_fwd(x, lab, 1e-4, nthreads=16)
    _, _, st = L.ce_zloss_forward(logits.detach(), labels, 1e-4)
    assert_bits_equal(st.cpu().numpy(), st_r, "row statistics")
    assert_bits_equal(np.array([ce.item(), z.item()], np.float32), np.array([ce_r, z_r], np.float32), "ce, z")
    rows = slice(4000, 4064)
    g_r = orc.ce_zloss_bwd(x[rows], lab[rows], st_r[:, rows], 1e-4, n_total=N, nthreads=16)
    assert_bits_equal(logits.grad[rows].float().cpu().numpy(), g_r, "logit gradient rows 4000..4063")


def _edge_rows(x, rng):
    """Rows that leave the window of the table form: zeros, subnormals, infinities, NaN, huge and tiny values, a row
    without a positive value, one of -inf alone, one of equal values."""
    V = x.shape[1]
    x[1, ::7] = 0.0
    x[2, V // 2] = -0.0
    x[3] *= 2.0 ** -20
    x[4] = -np.abs(x[4]) - 2.0 ** -10
    x[5, 5], x[5, V - 1] = np.inf, 300.0
    x[6, rng.integers(0, V, 3)] = -np.inf
    x[7, V - 2] = np.nan
    x[8] = -np.inf
    x[9] = 1.5
    x[10, :40] = 1e-40
    x[11] = rng.standard_normal(V) * 400
    x[12] = -0.0
    return x


@pytest.mark.parametrize("N,V,dtype", [
    (300, 16384, "bf16"),  # the table form's shortest row; more rows than CUs
    (17, 16408, "bf16"),   # a last chunk of 24
    (14, 131072, "bf16"),  # the longest row
    (17, 16376, "bf16"),   # just under the table form
    (17, 20001, "bf16"),   # unaligned rows, sixteen waves
    (15, 2048, "f32"),     # one wave per row, whole tiles
    (15, 2049, "bf16"),    # four waves, one logit past a tile
    (15, 16388, "f32"),    # sixteen waves
    (33000, 40, "f32"),    # more rows than workgroups
])
def test_loss_forms_and_edge_rows(N, V, dtype):
    """Every form of the kernels at the edges of its range, with rows that hold values outside the table's window:
    statistics, scalars and gradient against the oracle (NaN where the oracle has NaN)."""
    from attn_util import assert_bits_equal_nan_class as eq

    print(f"loss forms N={N} V={V} {dtype}", flush=True)
    x, lab = _inputs(N, V, dtype, seed=N + V, scale=2.0)
    x = _edge_rows(x, np.random.default_rng(V))
    if dtype == "bf16":
        x = synthetic.round_to_bf16(x)
    lab[5], lab[7] = 5, V - 2
    labels = torch.from_numpy(lab).to(DEV)
    logits = _gpu(x, dtype)
    with np.errstate(all="ignore"):
        ce_r, z_r, st_r = orc.ce_zloss_fwd(x, lab, 1e-4, nthreads=8)
        g_r = orc.ce_zloss_bwd(x, lab, st_r, 1e-4, gce=2.0, gz=3.0, out_bf16=dtype == "bf16", nthreads=8)
    ce, z, st = L.ce_zloss_forward(logits, labels, 1e-4)
    g = L.ce_zloss_backward(logits, labels, st, torch.tensor(2.0, device=DEV), torch.tensor(3.0, device=DEV), 1e-4)
    torch.cuda.synchronize()
    eq(st.cpu().numpy(), st_r, "row statistics")
    eq(np.array([ce.item(), z.item()], np.float32), np.array([ce_r, z_r], np.float32), "ce, z")
    eq(g.float().cpu().numpy(), g_r, "logit gradient")


@pytest.mark.parametrize("N,V,dtype", [
    (24, 16384, "bf16"),  # the table form
    (24, 4096, "bf16"),   # the general form, 16-byte vectors
    (24, 4099, "f32"),    # element by element
])
def test_backward_from_a_maximum_below_the_logits(N, V, dtype):
    """ce_zloss_backward takes the caller's statistics: with a stored maximum below some logits (or above all of them,
    infinite or NaN) exp(x - m) is still the correctly rounded one, in every form of the kernel."""
    from attn_util import assert_bits_equal_nan_class as eq

    print(f"loss backward, maximum below the logits N={N} V={V} {dtype}", flush=True)
    x, lab = _inputs(N, V, dtype, seed=N + V, scale=2.0)
    x = _edge_rows(x, np.random.default_rng(V))
    if dtype == "bf16":
        x = synthetic.round_to_bf16(x)
    with np.errstate(all="ignore"):
        st = orc.ce_zloss_fwd(x, lab, 1e-4)[2]
        st[0] -= np.resize(np.array([0.5, 3.0, 60.0, 100.0, -2.0], np.float32), N)
        st[0, 13], st[0, 14], st[0, 15] = np.nan, np.inf, -np.inf
        g_r = orc.ce_zloss_bwd(x, lab, st, 1e-4, gce=2.0, gz=3.0, out_bf16=dtype == "bf16")
    assert np.isinf(g_r).any() and (st[0] < x.max(1)).any()
    two, three = torch.tensor(2.0, device=DEV), torch.tensor(3.0, device=DEV)
    g = L.ce_zloss_backward(_gpu(x, dtype), torch.from_numpy(lab).to(DEV), torch.from_numpy(st).to(DEV), two, three, 1e-4)
    torch.cuda.synchronize()
    eq(g.float().cpu().numpy(), g_r, "logit gradient")
