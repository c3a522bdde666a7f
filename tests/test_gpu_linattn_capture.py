"""Linear-attention calls recorded into graphs: what check_status() reports of
their replays, and that graphs and eager calls never meet in a workspace."""

import pytest
import torch

from kernelforge_amd import _lib
from kernelforge_amd.SANA_LinearAttention import check_status, custom, linear_attention
from kernelforge_amd.SANA_LinearAttention.fused import litela_fused_attention

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


def capture(stream, *calls):
    """A graph of linear_attention calls on ``stream``, whose pool first held a
    tensor of nonzero bytes."""
    stream.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        junk = torch.full((32 << 20,), 1, dtype=torch.uint8, device=DEV)
        del junk
        outs = [linear_attention(qkv, H, D) for qkv, H, D in calls]
    return graph, outs


def test_eager_call_on_the_capture_stream():
    """An eager call on the stream of a capture, with more (batch, head pair)
    groups than the captured calls cleared, before and after replays."""
    small, other = packed(1, 300, 4, 32, seed=2), packed(1, 300, 3, 64, seed=3)
    big = packed(2, 512, 36, 32, seed=4)
    want = [linear_attention(x, H, D) for x, H, D in ((small, 4, 32), (other, 3, 64), (big, 36, 32))]
    check_status()
    stream = torch.cuda.Stream()
    for first, D in (((other, 3, 64), 64), ((small, 4, 32), 32)):
        print(f"captured D={D}", flush=True)
        graph, outs = capture(stream, first)
        for replays in (0, 1, 2):
            with torch.cuda.stream(stream):
                for _ in range(replays):
                    graph.replay()
                got = linear_attention(big, 36, 32)
            torch.cuda.synchronize()
            assert torch.equal(got, want[2])
            check_status()
        assert torch.equal(outs[0], want[1] if D == 64 else want[0])


def test_graphs_keep_their_workspaces():
    """Replays after a larger eager call on the capture stream and tensors in
    the memory it may have freed, after another graph of the stream is gone,
    and of two graphs at once on two streams."""
    a, b = packed(1, 2048, 8, 32, seed=5), packed(2, 1500, 24, 32, seed=6)
    large = packed(2, 4096, 70, 32, seed=7)
    want_a, want_b = linear_attention(a, 8, 32), linear_attention(b, 24, 32)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        linear_attention(a, 8, 32)
    gone, _ = capture(stream, (a, 8, 32))
    ga, (out_a,) = capture(stream, (a, 8, 32))
    gb, (out_b,) = capture(stream, (b, 24, 32))
    with torch.cuda.stream(stream):
        linear_attention(large, 70, 32)
    del gone
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    filler = [torch.full((1 << 20,), 3, dtype=torch.uint8, device=DEV) for _ in range(64)]
    other = torch.cuda.Stream()
    for rep in range(4):
        print(f"replay {rep}", flush=True)
        out_a.fill_(float("nan"))
        out_b.fill_(float("nan"))
        stream.wait_stream(torch.cuda.current_stream())
        other.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            ga.replay()
        with torch.cuda.stream(other):
            gb.replay()
        torch.cuda.synchronize()
        assert torch.equal(out_a, want_a) and torch.equal(out_b, want_b)
        assert all(bool((f == 3).all()) for f in filler)
        check_status()


def test_fused_projection_graphs_on_two_streams():
    """Graphs of the fused projection path captured on one stream and replayed
    at once on two, after a larger eager call on the capture stream."""
    def inputs(B, N, H, seed):
        g = torch.Generator().manual_seed(seed)
        x = torch.randn((B, N, 32 * H), generator=g)
        w = torch.randn((96 * H, 32 * H), generator=g) * (32 * H) ** -0.5
        return x.to(torch.bfloat16).to(DEV), w.to(torch.bfloat16).to(DEV), H

    def run(x, w, H):
        return litela_fused_attention(x, w, None, H)

    cases = [inputs(1, 700, 12, 1), inputs(2, 900, 9, 2)]
    large = inputs(2, 2048, 36, 3)
    want = [run(*c) for c in cases]
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        run(*cases[0])
    graphs, outs = [], []
    for case in cases:
        graphs.append(torch.cuda.CUDAGraph())
        with torch.cuda.graph(graphs[-1], stream=stream):
            outs.append(run(*case))
    with torch.cuda.stream(stream):
        run(*large)
    torch.cuda.synchronize()
    streams = [stream, torch.cuda.Stream()]
    for rep in range(4):
        print(f"replay {rep}", flush=True)
        for out in outs:
            out.fill_(float("nan"))
        for s, graph in zip(streams, graphs):
            s.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(s):
                graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(out, w) for out, w in zip(outs, want))
