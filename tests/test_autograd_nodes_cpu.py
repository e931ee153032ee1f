"""What the native autograd nodes refuse before any launch (no GPU needed: the checks stand before the first device
call)."""

from __future__ import annotations

import pytest
import torch

from open_transformers_amd import _lib


@pytest.mark.parametrize("rows", [0, 4])
def test_an_empty_width_is_refused(rows):
    nodes = _lib.autograd()
    x = torch.empty(rows, 0, dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="last dimension"):
        nodes.rms_norm(x, torch.empty(0, dtype=torch.bfloat16), 1e-5)
    with pytest.raises(ValueError, match="last dimension"):
        nodes.swiglu(x)


def test_a_weight_of_another_size_or_device_is_refused():
    """The kernels take the weight's size from the input: a smaller one would be read past its end."""
    nodes = _lib.autograd()
    x = torch.zeros(128, 256, dtype=torch.bfloat16)
    w = torch.zeros(128, 256, dtype=torch.bfloat16)
    for bad in (w[:, :128], w[:, :128].contiguous(), torch.zeros(128, 288, dtype=torch.bfloat16), w.view(-1)):
        with pytest.raises(ValueError, match="weight"):
            nodes.linear(x, bad)
    for bad in (w[0, :128], w[:1, :128], w):
        with pytest.raises(ValueError, match="weight"):
            nodes.rms_norm(x, bad, 1e-5)
    for call in (lambda: nodes.linear(x, w.to("meta")), lambda: nodes.rms_norm(x, w[0].to("meta"), 1e-5),
                 lambda: nodes.rope_heads(x.view(1, 32, 8, 128), torch.zeros(32, 64), torch.zeros(32, 64, device="meta"))):
        with pytest.raises(RuntimeError, match="same device"):
            call()
