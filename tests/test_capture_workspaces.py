"""Workspaces under graph capture (no GPU): the allocation rule with the device
calls replaced.  A captured call's workspace never enters the table that eager
calls use, and an eager call's never enters a graph."""

import pytest
import torch

from kernelforge_amd import _lib
from kernelforge_amd.SANA_LinearAttention import custom, fused

CPU = torch.device("cpu", 0)


class Calls:
    """Records the C calls made on a workspace."""

    def __init__(self):
        self.made = []

    def __getattr__(self, name):
        def call(ptr, *args):
            self.made.append((name, ptr.value))
            return 0
        return call


@pytest.fixture
def device(monkeypatch):
    """(capturing flag setter, recorded C calls) of a pretended stream 77."""
    state = dict(capturing=False)
    calls = Calls()
    monkeypatch.setattr(torch._C, "_cuda_isCurrentStreamCapturing", lambda: state["capturing"])
    monkeypatch.setattr(_lib, "current_stream", lambda index: 77)
    monkeypatch.setattr(_lib, "load", lambda: calls)
    return lambda on: state.update(capturing=on), calls


def test_linear_attention_workspaces(device, monkeypatch):
    monkeypatch.setattr(custom, "_workspaces", {})
    monkeypatch.setattr(custom, "_captured_devices", set())
    capturing, calls = device
    size = 2 << 20
    shape = (1, 4, 32, _lib.KF_BF16)

    capturing(True)
    captured = custom._workspace(CPU, size, shape)
    assert not custom._workspaces and custom._captured_devices == {0}
    assert calls.made == [("kf_linattn_capture_init", captured.data_ptr())]

    capturing(False)
    captured.fill_(255)
    eager = custom._workspace(CPU, size, shape)
    assert eager.data_ptr() != captured.data_ptr() and not eager.any()
    assert custom._workspace(CPU, 1 << 20, shape) is eager
    assert len(calls.made) == 1  # eager calls find their control words zero

    capturing(True)
    again = custom._workspace(CPU, 1 << 20, shape)
    assert again.data_ptr() not in (eager.data_ptr(), captured.data_ptr())
    assert list(custom._workspaces.values()) == [eager]


def test_fused_projection_workspaces(device, monkeypatch):
    monkeypatch.setattr(fused, "_workspaces", {})
    capturing, _ = device
    capturing(True)
    captured = fused._workspace(CPU, 4096)
    assert captured.numel() >= 4096 and not fused._workspaces
    capturing(False)
    eager = fused._workspace(CPU, 8192)
    assert fused._workspace(CPU, 4096) is eager
    capturing(True)
    assert fused._workspace(CPU, 4096).data_ptr() not in (eager.data_ptr(), captured.data_ptr())
    assert list(fused._workspaces.values()) == [eager]
