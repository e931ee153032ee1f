"""The four-waves-per-block attention kernels (forward, dK/dV, dQ), byte for byte,
at the edges of their tiles and on both sides of every limit of the launcher's
choice: small shapes against the CPU oracle; bf16 at the limits against the
one-wave-per-block kernels; binary32 at the limits, whose forward and dK/dV have
no other form, in both widths of the tile kernels against each other and with two
(batch, head group) slices against the oracle.

In the default launch the choice goes by the number of 32-row blocks over all
heads (256 compute units: forward 256, 512 and 1024 blocks, dK/dV 128, 512 and
2048 key blocks, dQ 512, 1024 and 2048); variants 1, 2 and 3 go by no limit (3 is
the default launch without the tile kernels).  The comparison is exact: all forms
are the same serial folds.
"""
from __future__ import annotations

import pytest
import torch

from attn_util import assert_bits_equal, gpu_fwd_bwd, make, oracle_fwd_bwd
from open_transformers_amd.nn import flash_attention as fa
from oracle import oracle as orc

pytestmark = pytest.mark.gpu
NAMES = ("o", "lse", "dq", "dk", "dv")

# (B, H, Hkv, S, D, window): one block; odd block counts (the last pair of key or query blocks is half empty); a window
# of one block, of an odd number of blocks and longer than the sequence; query groups
SMALL = [(1, 1, 1, 32, 64, 0), (1, 2, 1, 64, 128, 0), (2, 3, 1, 96, 128, 32), (1, 2, 2, 160, 64, 96),
         (1, 4, 2, 224, 128, 64), (1, 2, 1, 96, 64, 320), (1, 1, 1, 288, 128, 0), (1, 8, 2, 224, 128, 0),
         (1, 4, 1, 96, 64, 0)]


@pytest.mark.parametrize("shape", SMALL, ids=[f"s{i}" for i in range(len(SMALL))])
@pytest.mark.parametrize("form", ["f32-0", "f32-1", "f32-2", "f32-3", "bf16-0", "bf16-0-cache", "bf16-3", "bf16-3-cache"])
def test_gpu_tile_small(shape, form):
    B, H, Hkv, S, D, window = shape
    bf16 = form.startswith("bf16")
    variant = int(form.split("-")[1])
    print(form, shape, flush=True)
    inp = make(B, H, Hkv, S, D, dtype="bf16" if bf16 else "f32", seed=S + D, qk_scale=3.0)
    got = gpu_fwd_bwd(inp, window, bf16, variant=variant, score_cache=form.endswith("cache"))
    ref = oracle_fwd_bwd(inp, window, bf16)
    for n in NAMES:
        assert_bits_equal(got[n], ref[n], n)


# block counts over all heads on either side of a limit: (B, H, Hkv, S, D, window)
LIMITS = [(1, 16, 8, 512, 128, 64), (1, 16, 8, 544, 128, 64), (1, 16, 16, 1024, 64, 0), (1, 16, 16, 1056, 64, 0),
          (1, 16, 16, 1024, 128, 96), (1, 16, 16, 1056, 128, 96), (1, 32, 32, 1024, 128, 0), (1, 32, 32, 1056, 128, 0),
          (2, 32, 16, 1024, 64, 64), (2, 32, 32, 1024, 128, 64), (2, 33, 33, 1024, 128, 64), (1, 32, 2, 1024, 128, 256),
          # past every limit, an odd number of blocks: the one-wave kernels' paired and head-grouped workgroups
          (4, 16, 16, 2080, 128, 0), (4, 16, 4, 2080, 128, 0), (4, 16, 4, 2080, 128, 512)]


@pytest.mark.parametrize("shape", LIMITS, ids=[f"l{i}" for i in range(len(LIMITS))])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_gpu_tile_choice(shape, dtype):
    """Variants 0, 1, 2 and 3, with the scores recomputed and (bf16) read from the cache of another variant's forward;
    binary32: the first and the last head group against the oracle besides (heads are independent)."""
    B, H, Hkv, S, D, window = shape
    print(dtype, shape, flush=True)
    T = torch.float32 if dtype == "f32" else torch.bfloat16
    g = torch.Generator(device="cuda").manual_seed(S + H)
    q, k, v, do = (torch.randn(B, h, S, D, device="cuda", generator=g).to(T) for h in (H, Hkv, Hkv, H))
    o, lse = fa.flash_attention_forward(q, k, v, window, variant=2)
    ref = fa.flash_attention_backward(q, k, v, o, lse, do, window, variant=2)
    for variant in (0, 1, 3):
        o2, lse2 = fa.flash_attention_forward(q, k, v, window, variant=variant)
        assert torch.equal(o, o2) and torch.equal(lse, lse2), variant
        for a, b, n in zip(ref, fa.flash_attention_backward(q, k, v, o, lse, do, window, variant=variant), NAMES[2:]):
            assert torch.equal(a, b), (n, variant)
    if dtype == "f32":
        G = H // Hkv
        for i, kv in ((0, 0), (B - 1, Hkv - 1)):
            qs = slice(G * kv, G * kv + G)
            part = {n: t[i:i + 1, s].cpu().numpy() for n, t, s in
                    (("q", q, qs), ("k", k, slice(kv, kv + 1)), ("v", v, slice(kv, kv + 1)), ("do", do, qs))}
            want = oracle_fwd_bwd(part, window, False)
            for n, t, s in zip(NAMES, (o, lse, *ref), (qs, qs, qs, slice(kv, kv + 1), slice(kv, kv + 1))):
                assert_bits_equal(t[i:i + 1, s].cpu().numpy(), want[n], f"{n} of head group {kv}")
    if dtype == "bf16":
        sc = [fa.flash_attention_forward_sc(q, k, v, window, variant=x) for x in (0, 2)]
        for a, b in zip(*sc):
            assert torch.equal(a, b)
        for variant in (0, 3):
            for a, b, n in zip(ref, fa.flash_attention_backward(q, k, v, o, lse, do, window, variant=variant,
                                                                score_cache=sc[1][2]), NAMES[2:]):
                assert torch.equal(a, b), (n, variant, "cache")


@pytest.mark.parametrize("shape", LIMITS, ids=[f"l{i}" for i in range(len(LIMITS))])
def test_gpu_tile_choice_int8pv(shape):
    """The int8-PV forward with its score cache, variants 0, 1, 2 and 3, and the first and the last head group's O and LSE
    against the oracle (heads are independent).  Some rows have scores so far apart that a block's probabilities are all
    +0 or below the step's normal range."""
    B, H, Hkv, S, D, window = shape
    print(shape, flush=True)
    g = torch.Generator(device="cuda").manual_seed(S + D)
    q, k, v = (torch.randn(B, h, S, D, device="cuda", generator=g).to(torch.bfloat16) for h in (H, Hkv, Hkv))
    q[:, :, 5::7] *= 12.0
    ref = fa.int8pv_flash_attention_forward_sc(q, k, v, window, variant=2)
    for variant in (0, 1, 3):
        for a, b in zip(ref, fa.int8pv_flash_attention_forward_sc(q, k, v, window, variant=variant)):
            assert torch.equal(a, b), variant
    G = H // Hkv
    for i, kv in ((0, 0), (B - 1, Hkv - 1)):
        qs = slice(G * kv, G * kv + G)
        part = [t[i:i + 1, s].float().cpu().numpy() for t, s in ((q, qs), (k, slice(kv, kv + 1)), (v, slice(kv, kv + 1)))]
        for t, want, n in zip(ref, orc.attn_fwd_int8pv(*part, window=window), NAMES):
            assert_bits_equal(t[i:i + 1, qs].float().cpu().numpy(), want, f"{n} of head group {kv}")


def test_more_workgroups_than_a_launch_row_holds():
    """A binary32 forward of 2^23 + 1 blocks in the sixteen-query form: 2^24 + 2 workgroups of 256 threads, more than one
    launch holds along x.  Heads from both rows of the grid against a call of those heads alone (they share one KV head)."""
    H = (1 << 23) + 1
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < 160 << 30:
        pytest.skip("needs 160 GiB of free device memory")
    print(f"binary32 forward of {H} heads", flush=True)
    g = torch.Generator(device="cuda").manual_seed(9)
    few = [0, 1, 12345, H // 2, H - 2, H - 1]
    qf, k, v = (torch.randn(1, n, 32, 64, device="cuda", generator=g) for n in (len(few), 1, 1))
    q = torch.zeros(1, H, 32, 64, device="cuda")
    q[:, few] = qf
    o, lse = fa.flash_attention_forward(q, k, v, variant=2)
    want_o, want_lse = fa.flash_attention_forward(qf, k, v, variant=2)
    got_o, got_lse = o[:, few], lse[:, few]
    same = torch.equal(got_o, want_o) and torch.equal(got_lse, want_lse)
    plain = torch.equal(o[:, 7], o[:, H - 5]) and torch.equal(lse[:, 7], lse[:, H - 5])  # heads of zero queries
    del q, o, lse
    torch.cuda.empty_cache()
    assert same and plain
