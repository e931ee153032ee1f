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
