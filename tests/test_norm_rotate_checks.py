"""The checks of LiteLA's q/k norm and rotary step before any kernel (no GPU): the
one-pass kernel takes raw pointers, so what the row norm refuses must not reach it."""

import pytest
import torch

from kernelforge_amd import _lib
from kernelforge_amd.SANA_LinearAttention import modules


class NoCalls:
    def __getattr__(self, name):
        raise AssertionError(f"{name} reached")


@pytest.fixture
def no_launch(monkeypatch):
    monkeypatch.setattr(_lib, "load", lambda: NoCalls())
    monkeypatch.setattr(_lib, "stream_of", lambda t: None)


def rotate(qw, kw):
    qkv = torch.zeros(1, 4, 3, 32, dtype=torch.bfloat16)
    modules._norm_rotate_(qkv, 1, 32, qw, kw, 1e-5, None)


def test_weights_off_the_gpu_are_refused(no_launch):
    with pytest.raises(ValueError, match="HIP"):
        rotate(torch.ones(32), torch.ones(32))


@pytest.mark.parametrize("shapes", [((32, 1), (32,)), ((32,), (1, 32)), ((31,), (32,)), ((32,), (64,))])
def test_weights_of_another_shape_are_refused(no_launch, monkeypatch, shapes):
    """With the device check passed (every tensor here is on the CPU)."""
    monkeypatch.setattr(_lib, "require_gpu", lambda *tensors: None)
    with pytest.raises((ValueError, AssertionError)) as e:
        rotate(*(torch.ones(s) for s in shapes))
    # A valid q weight is normalised with before the k weight is looked at.
    assert "shape" in str(e.value) or "kf_rmsnorm_fwd_strided reached" in str(e.value)
