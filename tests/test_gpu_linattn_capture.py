"""Linear-attention calls recorded into graphs: what check_status() reports of
their replays."""

import pytest
import torch

from kernelforge_amd import _lib
from kernelforge_amd.SANA_LinearAttention import check_status, custom, linear_attention

pytestmark = pytest.mark.gpu
DEV = "cuda"


def packed(B, N, H, D, seed, dtype=torch.bfloat16):
    g = torch.Generator().manual_seed(seed)
    return torch.randn((B, N, 3, H * D), generator=g).to(dtype).to(DEV)


class FirstCallGivesUp:
    """The library, with the poll limit of the first kf_linattn_fwd cut to two
    polls (kfm_linattn_fwd_spin): members that arrive before the rest of their
    group stop waiting and write NaN."""

    def __init__(self, lib):
        self.lib, self.calls = lib, 0

    def __getattr__(self, name):
        return getattr(self.lib, name)

    def kf_linattn_fwd(self, *args):
        self.calls += 1
        if self.calls == 1:
            return self.lib.kfm_linattn_fwd_spin(*args[:-1], 2, args[-1])
        return self.lib.kf_linattn_fwd(*args)


def test_check_status_reports_an_earlier_node(monkeypatch):
    """A graph of three calls, the first of which gives up: the later nodes and
    later replays must not hide the report, which is raised once."""
    qkv = packed(1, 2048, 4, 32, seed=1)
    want = linear_attention(qkv, 4, 32, splits=8)
    check_status()
    lib = FirstCallGivesUp(_lib.load())
    graph = torch.cuda.CUDAGraph()
    with monkeypatch.context() as m:
        m.setattr(custom._lib, "load", lambda: lib)
        with torch.cuda.graph(graph):
            outs = [linear_attention(qkv, 4, 32, splits=8) for _ in range(3)]
    assert lib.calls == 3
    reported = 0
    for rep in range(5):
        print(f"replay {rep}", flush=True)
        graph.replay()
        torch.cuda.synchronize()
        gave_up = bool(torch.isnan(outs[0]).any())
        assert torch.equal(outs[1], want) and torch.equal(outs[2], want)
        if gave_up:
            reported += 1
            if rep % 2:
                graph.replay()  # whatever it does, the report above stands
            with pytest.raises(RuntimeError, match="stopped waiting"):
                check_status()
        check_status()
    assert reported, "no member stopped waiting at a two-poll limit"
    assert torch.equal(linear_attention(qkv, 4, 32, splits=8, check=True), want)
