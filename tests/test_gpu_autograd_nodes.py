"""The native autograd nodes as autograd sees them: saved-tensor hooks reach every saved tensor, a saved input changed
in place is refused, a gradient that nobody asks for is not computed, an unused output counts as a zero gradient, and
non-contiguous and expanded upstream gradients give the bytes of contiguous ones; other streams and threads, traces, and
the transforms that have no rule for a node and refuse it."""

from __future__ import annotations

import threading

import pytest
import torch

from open_transformers_amd.nn import flash_attention as fa
from open_transformers_amd.nn import functional as F
from open_transformers_amd.nn.embedding import embedding
from open_transformers_amd.nn.flash_attention import causal_flash_attention, int8pv_causal_flash_attention
from open_transformers_amd.nn.layer import rope_tables
from open_transformers_amd.nn.loss import fused_ce_z_loss

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _rand(*shape, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed + sum(shape))
    return torch.randn(shape, device=DEV, generator=g).bfloat16().requires_grad_()


def _cases():
    cos, sin = (t.to(DEV) for t in rope_tables(64, 64, 10000.0))
    q, k, v = _rand(1, 4, 64, 64), _rand(1, 2, 64, 64, seed=1), _rand(1, 2, 64, 64, seed=2)
    ids = torch.arange(64, device=DEV) % 16
    return {  # name: (call, inputs, tensors the node saves)
        "linear": (F.linear, (_rand(128, 128), _rand(256, 128)), 2),
        "rms_norm": (lambda x, w: F.rms_norm(x, w, 1e-5), (_rand(64, 128), _rand(128)), 3),
        "silu": (F.silu, (_rand(33, 7),), 1),
        "swiglu": (F.swiglu, (_rand(8, 64),), 1),
        "rope_heads": (lambda x: F.rope_heads(x, cos, sin), (_rand(2, 64, 4, 64),), 2),
        "heads": (F.heads, (_rand(2, 64, 4, 64),), 0),
        "embedding": (lambda w: embedding(ids, w), (_rand(16, 64),), 1),
        "attention": (causal_flash_attention, (q, k, v), 6),
        "attention_int8pv": (int8pv_causal_flash_attention, (q, k, v), 6),
        "loss": (lambda x: fused_ce_z_loss(x, ids, 1e-4)[0], (_rand(64, 100),), 3),
    }


NAMES = ["linear", "rms_norm", "silu", "swiglu", "rope_heads", "heads", "embedding", "attention", "attention_int8pv",
         "loss"]


def _bits(t):
    return t.contiguous().view(torch.int16 if t.dtype == torch.bfloat16 else torch.int32)


@pytest.mark.parametrize("name", NAMES)
def test_hooks_partial_and_strided_gradients(name):
    print(f"autograd node {name}", flush=True)
    call, inputs, nsaved = _cases()[name]
    y = call(*inputs)
    dy = torch.randn(y.shape, device=DEV).to(y.dtype)
    ref = torch.autograd.grad(y, inputs, dy)

    packed = []

    def pack(t):
        packed.append(t)
        return t.cpu()

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.to(DEV)):
        y2 = call(*inputs)
    assert len(packed) == nsaved
    for a, b in zip(torch.autograd.grad(y2, inputs, dy), ref):
        assert torch.equal(_bits(a), _bits(b))

    for i in range(len(inputs)):  # one input at a time
        args = [t if j == i else t.detach() for j, t in enumerate(inputs)]
        (g,) = torch.autograd.grad(call(*args), [inputs[i]], dy)
        assert torch.equal(_bits(g), _bits(ref[i]))

    if y.dim() >= 2:  # a transposed upstream gradient of the same values
        strided = dy.transpose(-1, -2).contiguous().transpose(-1, -2)
        for a, b in zip(torch.autograd.grad(call(*inputs), inputs, strided), ref):
            assert torch.equal(_bits(a), _bits(b))
        expanded = torch.ones(1, device=DEV, dtype=y.dtype).expand(y.shape)
        for a, b in zip(torch.autograd.grad(call(*inputs), inputs, expanded),
                        torch.autograd.grad(call(*inputs), inputs, torch.ones_like(y))):
            assert torch.equal(_bits(a), _bits(b))
    with torch.no_grad():
        assert torch.equal(_bits(call(*inputs)), _bits(y.detach()))
    torch.cuda.synchronize()


@pytest.mark.parametrize("name", ["linear", "rms_norm", "silu", "swiglu", "attention", "loss"])
def test_saved_input_changed_in_place_is_refused(name):
    call, inputs, _ = _cases()[name]
    x = inputs[0].detach().clone().requires_grad_()
    y = call(x, *inputs[1:])
    with torch.no_grad():
        x.add_(1.0)
    with pytest.raises(RuntimeError, match="inplace"):
        torch.autograd.grad(y.sum(), [x])


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("name", NAMES)
def test_a_trace_replays_the_operator(name, grad):
    """torch.jit.trace, recorded with inputs that do and do not require gradients: the traced call on other values gives
    the operator's bytes and gradients."""
    call, inputs, _ = _cases()[name]
    print(f"autograd node {name}: traced", flush=True)
    traced = torch.jit.trace(call, tuple(t.detach().requires_grad_(grad) for t in inputs), check_trace=False)
    args = [(t.detach() * 0.5).requires_grad_() for t in inputs]
    y, ref = traced(*args), call(*args)
    assert torch.equal(_bits(y.detach()), _bits(ref.detach()))
    dy = torch.randn(y.shape, device=DEV).to(y.dtype)
    for a, b in zip(torch.autograd.grad(y, args, dy), torch.autograd.grad(ref, args, dy)):
        assert torch.equal(_bits(a), _bits(b))


@pytest.mark.parametrize("name", [n for n in NAMES if n != "heads"])
def test_a_saved_tensor_that_comes_back_changed_is_refused(name):
    """A saved-tensor hook may hand back anything, and the kernels see only addresses: every saved tensor that comes back
    shorter, longer or in another type is a ValueError, and one of other strides is either that or read correctly."""
    call, inputs, nsaved = _cases()[name]
    ref = torch.autograd.grad(call(*inputs).sum(), inputs)

    def backward(which, change):
        count = iter(range(nsaved))

        def unpack(packed):
            i, t = packed
            return change(t) if i == which else t

        with torch.autograd.graph.saved_tensors_hooks(lambda t: (next(count), t.detach()), unpack):
            y = call(*inputs)
        return torch.autograd.grad(y.sum(), inputs)

    other = {torch.bfloat16: torch.float32, torch.float32: torch.bfloat16, torch.int64: torch.int32}
    changes = {
        "shorter": lambda t: t[: t.shape[0] - 1].contiguous(),
        "narrower": lambda t: t[..., : t.shape[-1] - 1].contiguous(),
        "another type": lambda t: t.to(other[t.dtype]),
    }
    for which in range(nsaved):
        for what, change in changes.items():
            if (name, which, what) == ("loss", 0, "another type"):
                continue  # the loss takes logits of either type
            print(f"autograd node {name}: saved tensor {which} {what}", flush=True)
            with pytest.raises((ValueError, RuntimeError)) as err:
                backward(which, change)
            # the loss's logits of another row count or width are refused as a gradient of the wrong shape
            assert isinstance(err.value, ValueError) or (name, which) == ("loss", 0), err.value
        strided = lambda t: t.transpose(-1, -2).contiguous().transpose(-1, -2) if t.dim() > 1 else t[:, None].expand(
            -1, 2).contiguous()[:, 0]
        try:
            got = backward(which, strided)
        except ValueError as err:
            assert name.startswith("attention") and "contiguous" in str(err)
        else:
            for a, b in zip(got, ref):
                assert torch.equal(_bits(a), _bits(b)), f"saved tensor {which} with other strides"
    torch.cuda.synchronize()


def _forward_backward(call, inputs, dy):
    args = [t.detach().requires_grad_() for t in inputs]
    y = call(*args)
    return [y.detach(), *torch.autograd.grad(y, args, dy)]


@pytest.mark.parametrize("name", NAMES)
def test_side_streams_and_threads(name):
    """Forward and backward on another stream, and on two threads with a stream each at once, the memory that the nodes
    take being used again at once by their own next calls: the bytes of the default stream."""
    print(f"autograd node {name}: streams and threads", flush=True)
    call, inputs, _ = _cases()[name]
    y = call(*inputs)
    dy = torch.randn(y.shape, device=DEV).to(y.dtype)
    ref = _forward_backward(call, inputs, dy)
    torch.cuda.synchronize()
    got = [[], []]

    def work(out):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for _ in range(8):
                out.append([t.clone() for t in _forward_backward(call, inputs, dy)])
        stream.synchronize()

    threads = [threading.Thread(target=work, args=(out,)) for out in got]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for out in got:
        assert len(out) == 8
        for run in out:
            for a, b in zip(run, ref):
                assert torch.equal(_bits(a), _bits(b))


@pytest.mark.parametrize("name", NAMES)
def test_transforms_without_a_rule_refuse(name):
    call, inputs, _ = _cases()[name]
    args = tuple(t.detach() for t in inputs)
    with pytest.raises(RuntimeError, match="functorch"):
        torch.func.vmap(call)(*[torch.stack([a, a]) for a in args])
    with pytest.raises(RuntimeError, match="functorch"):
        torch.func.grad(lambda *a: call(*a).sum())(*args)
    with torch.autograd.forward_ad.dual_level(), pytest.raises(RuntimeError, match="jvp"):
        call(*[torch.autograd.forward_ad.make_dual(a, a) for a in args])


@pytest.mark.parametrize("cache", [False, True])
@pytest.mark.parametrize("int8pv", [False, True])
def test_both_attention_nodes_save_the_same_tensors(int8pv, cache):
    """A checkpoint's first forward may run the Python node and its recompute the native one: the same tensors, in the
    same order, and the same result."""
    _, inputs, _ = _cases()["attention"]
    python = fa._Int8PVFlashAttention if int8pv else fa._CausalFlashAttention
    native = int8pv_causal_flash_attention if int8pv else causal_flash_attention
    saved = ([], [])

    def packing(out):
        def pack(t):
            out.append(t.detach().clone())
            return t

        return torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t)

    before = fa.set_score_cache(cache)
    try:
        with packing(saved[0]):
            a = python.apply(*inputs, 32, fa._score_cache_mode(*inputs))
        with packing(saved[1]):
            b = native(*inputs, window=32)
    finally:
        fa.set_score_cache(before)
    assert len(saved[0]) == len(saved[1]) == (6 if cache else 5)
    for x, y in zip((a.detach(), *saved[0]), (b.detach(), *saved[1])):
        assert x.shape == y.shape and x.dtype == y.dtype and torch.equal(_bits(x), _bits(y))
