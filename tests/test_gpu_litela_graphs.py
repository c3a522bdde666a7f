"""Two LiteLA blocks captured on one stream, a workspace of its own for each
captured call: either graph may be replayed first, and often."""

import pytest
import torch

from kernelforge_amd.SANA_LinearAttention import CUDAGraphJointLiteLA, optimized_joint_litela

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,C", [(1024, 1152), (300, 384)])
def test_second_graph_first(N, C):
    mods, graphs, xs, want = [], [], [], []
    for seed in range(2):
        torch.manual_seed(seed)
        with torch.device("cuda"):
            m = optimized_joint_litela(C, C, batch=1, seq_len=N, dtype=torch.bfloat16)
        m = m.to(torch.bfloat16)
        x = torch.randn(1, N, C, device="cuda").to(torch.bfloat16)
        with torch.inference_mode():
            want.append(m(x))
        mods.append(m)
        xs.append(x)
        graphs.append(CUDAGraphJointLiteLA(m))
    for i in (1, 0, 1, 1, 0):
        got = graphs[i](xs[i])
        torch.cuda.synchronize()
        assert torch.equal(got, want[i])
        with torch.inference_mode():  # eager work between replays
            assert torch.equal(mods[1 - i](xs[1 - i]), want[1 - i])
