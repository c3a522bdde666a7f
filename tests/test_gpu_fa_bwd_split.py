"""The split dK/dV backward (several workgroups per key tile, fp32 partial
sums joined in order): both kernels at every split against the unsplit kernel
and the fp64 gradients.

The splits only change the order of fp32 sums of the same products (relative
2^-24 per term) before the one rounding to 16 bits, so split and unsplit
results differ by at most one ulp (2^-7 relative for bf16, 2^-10 for fp16) plus
1e-5 of the tensor's scale where products cancel; dQ is the same bit for bit.
"""

import pytest
import torch

from kernelforge_amd import _lib
from kernelforge_amd.flash_attention_jvp import flash_attention, flash_attention_backward
from oracle import fa as orc

pytestmark = pytest.mark.gpu
DEV = "cuda"
ULP = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}
TOL = {torch.float16: dict(atol=3e-3, rtol=1e-2), torch.bfloat16: dict(atol=3e-2, rtol=3e-2)}

# One tile, tile edges (128 / 256 / 512 keys, 64 rows), GQA groups whose runs
# cross heads, causal tiles with fewer units than splits, rows without a key,
# keys no row sees, and D > 128.
CASES = [(1, 1, 1, 2, 2, 64, True), (2, 130, 257, 4, 1, 128, False), (1, 300, 300, 8, 2, 72, True),
         (1, 65, 513, 2, 2, 32, True), (1, 71, 19, 4, 1, 96, True), (1, 200, 200, 4, 2, 256, True),
         (1, 640, 128, 2, 1, 64, False)]


def setup(case, dtype):
    B, Nq, Nk, Hq, Hkv, D, causal = case
    g = torch.Generator().manual_seed(D + Nq)
    q, k, v, cot = (torch.randn(s, generator=g).to(dtype).to(DEV)
                    for s in ((B, Nq, Hq, D), (B, Nk, Hkv, D), (B, Nk, Hkv, D), (B, Nq, Hq, D)))
    return (q, k, v, cot, *flash_attention(q, k, v, causal=causal, return_lse=True))


def forced(q, k, v, cot, out, lse, causal, blocks, splits):
    B, Nq, Hq, D = q.shape
    Nk, Hkv = k.shape[1:3]
    lib = _lib.load()
    stats = -(-lib.kf_fa_bwd_workspace_bytes(B, Nq, Hq, D) // 256) * 256
    nbytes = stats + 8 * splits * B * Nk * Hkv * D
    ws = torch.full((nbytes,), 255, device=DEV, dtype=torch.uint8)  # NaN partials
    grads = tuple(torch.full_like(x, float("nan")) for x in (q, k, v))
    rc = lib.kfm_fa_bwd_split(*map(_lib.ptr, (q, k, v, out, lse, cot, *grads, ws)), nbytes, B, Nq, Nk, Hq, Hkv, D,
                              D ** -0.5, int(causal), _lib.kf_dtype(q.dtype), blocks, splits, _lib.stream_of(q))
    _lib.check(rc, "kfm_fa_bwd_split")
    return grads


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", CASES)
def test_every_split(case, dtype):
    causal = case[-1]
    args = setup(case, dtype)
    leaves = tuple(x.cpu().double().requires_grad_() for x in args[:3])
    ref = torch.autograd.grad(orc.attention(*leaves, causal=causal), leaves, args[3].cpu().double())
    for blocks in (1, 2):
        base = forced(*args, causal, blocks, 1)
        for splits in (1, 2, 3, 16):
            got = forced(*args, causal, blocks, splits)
            assert torch.equal(got[0], base[0])
            for a, b, r in zip(got, base, ref):
                torch.testing.assert_close(a.cpu().double(), r, **TOL[dtype])
                scale = float(b.float().abs().max())
                torch.testing.assert_close(a.float(), b.float(), rtol=ULP[dtype], atol=1e-5 * scale)
            again = forced(*args, causal, blocks, splits)
            assert all(torch.equal(a, b) for a, b in zip(got, again))


@pytest.mark.parametrize("case", [(1, 700, 700, 8, 2, 128, True), (1, 1000, 1000, 2, 2, 64, False),
                                  (1, 124, 124, 32, 8, 80, False)])
def test_public_backward_on_small_grids(case):
    q, k, v, cot, out, lse = setup(case, torch.bfloat16)
    got = flash_attention_backward(cot, q, k, v, out, lse, causal=case[-1])
    leaves = tuple(x.cpu().double().requires_grad_() for x in (q, k, v))
    ref = torch.autograd.grad(orc.attention(*leaves, causal=case[-1]), leaves, cot.cpu().double())
    for a, r in zip(got, ref):
        torch.testing.assert_close(a.cpu().double(), r, **TOL[torch.bfloat16])
        assert float((a.cpu().double() - r).norm() / r.norm()) < 1e-2
