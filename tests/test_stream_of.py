"""The stream lookup of a launch (no GPU)."""

import pytest
import torch

from kernelforge_amd import _lib


def test_a_cpu_tensor_has_no_stream(monkeypatch):
    """Operators called with tensors on mixed devices reach the lookup with a
    CPU tensor; torch would give its device index -1 the current stream."""
    monkeypatch.setattr(_lib, "current_stream", lambda index: 77)
    with pytest.raises(ValueError, match="HIP"):
        _lib.stream_of(torch.empty(1))
