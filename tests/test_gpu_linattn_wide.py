"""Linear attention on the matrix cores for D = 16, 64, 128 and fp32 D = 32
(kernelforge_amd/csrc/linattn_wide.h): against the fp64 formula and against the
VALU kernels, which the same call reaches when its buffer is not 16-byte
aligned.

Both paths multiply exactly or in fp32 and sum in fp32, in different orders.
A sum of n fp32 terms in any order is within n 2^-24 of the terms' absolute
sum, and typically sqrt(n) 2^-24: at n <= 1200 tokens 2e-6, so 4e-6 (relative
2-norm) bounds the state, contraction and division together; a 16-bit result
adds half an ulp (2^-8 relative for bf16's 8 significant bits, 2^-11 for fp16's 11).
"""

import pytest
import torch

from kernelforge_amd.SANA_LinearAttention import attn_matmul, linear_attention

pytestmark = pytest.mark.gpu
DEV = "cuda"
BOUND = {torch.float32: 4e-6, torch.bfloat16: 4e-6 + 2.0 ** -8, torch.float16: 4e-6 + 2.0 ** -11}


def packed(B, N, H, D, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randn((B, N, 3, H * D), generator=g).to(dtype)


def exact(qkv, H, D, eps=1e-15):
    q, k, v = (t.double().unflatten(-1, (H, D)).transpose(1, 2) for t in qkv.unbind(2))
    q, k = q.relu(), k.relu()
    num = q @ (k.transpose(-1, -2) @ v)
    den = (q * k.sum(-2, keepdim=True)).sum(-1, keepdim=True)
    return (num / (den + eps)).transpose(1, 2).flatten(2)


def unaligned(t):
    """The same values at an address that is 2 or 4 bytes past a 16-byte boundary."""
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=DEV)
    out = flat[1:].view(t.shape)
    out.copy_(t)
    assert out.data_ptr() % 16 != 0 and out.is_contiguous()
    return out


def rel(a, b):
    return float((a.double() - b.double()).norm() / b.double().norm())


# One token, tile edges (32, 64 and 128 tokens per tile), several splits and
# runs, head counts that leave a group of 64 / D heads partly filled.
SIZES = [(1, 1, 1), (1, 31, 3), (2, 64, 5), (1, 129, 2), (3, 257, 4), (2, 1200, 7)]


@pytest.mark.parametrize("B,N,H", SIZES)
@pytest.mark.parametrize("dtype,D", [(dt, d) for dt in (torch.bfloat16, torch.float16, torch.float32)
                                     for d in (16, 64, 128)] + [(torch.float32, 32)])
def test_matches_exact_and_valu(B, N, H, dtype, D):
    qkv = packed(B, N, H, D, dtype, seed=N + D)
    want = exact(qkv, H, D)
    dev = qkv.to(DEV)
    for out_dtype in dict.fromkeys((torch.float32, dtype, torch.bfloat16)):
        got = linear_attention(dev, H, D, output_dtype=out_dtype)
        valu = linear_attention(unaligned(dev), H, D, output_dtype=out_dtype)
        assert rel(got.cpu(), want) <= BOUND[out_dtype]
        assert rel(got, valu) <= 2 * BOUND[out_dtype]  # both within the bound of the exact value
    again = linear_attention(dev, H, D, output_dtype=torch.float32)
    assert torch.equal(again, linear_attention(dev, H, D, output_dtype=torch.float32))


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 64), (torch.float32, 32), (torch.float16, 16),
                                     (torch.float32, 128)])
def test_transposed_output(dtype, D):
    B, N, H = 2, 300, 3
    qkv = packed(B, N, H, D, dtype, seed=D).to(DEV)
    q, k, v = (qkv[:, :, p].view(B, N, H, D).permute(0, 2, 3, 1) for p in range(3))
    out = attn_matmul(q, k.transpose(-1, -2), v)
    want = exact(qkv.cpu(), H, D).view(B, N, H, D).permute(0, 2, 3, 1)
    assert out.shape == (B, H, D, N) and rel(out.cpu(), want) <= BOUND[torch.float32]


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 64), (torch.float16, 64), (torch.float32, 32),
                                     (torch.bfloat16, 16), (torch.bfloat16, 128)])
def test_special_values_stay_in_their_heads(dtype, D):
    """Infinities and NaN in one head's q, k or v leave the other heads'
    results as they are and give what the VALU path gives in theirs."""
    B, N, H = 1, 150, 4
    clean = packed(B, N, H, D, dtype, seed=9).to(DEV)
    qkv = clean.clone()
    qkv[0, 3, 0, 1] = float("inf")        # head 0: q
    qkv[0, 5, 0, 2] = float("nan")
    qkv[0, 70, 1, D + 1] = float("inf")   # head 1: k
    qkv[0, 71, 1, D + 2] = float("nan")
    qkv[0, 9, 2, 2 * D + 1] = float("-inf")  # head 2: v
    got = linear_attention(qkv, H, D)
    valu = linear_attention(unaligned(qkv), H, D)
    assert torch.equal(torch.isnan(got), torch.isnan(valu))
    assert torch.equal(torch.isinf(got), torch.isinf(valu))
    fine = torch.isfinite(valu)
    assert rel(got[fine], valu[fine]) <= 2 * BOUND[torch.float32]
    assert torch.equal(got[..., 3 * D:], linear_attention(clean, H, D)[..., 3 * D:])


# Denominators whose reciprocal overflows or is subnormal, with quotients near 1:
# q and k are scaled so that z . relu(q), whose mean is 150 D E[relu^]^2 scale^2
# = 24 D scale^2 for normal values, is about 1e-41 or 1.2e38 (fp32 ends at
# 3.4e38).  A sum of 150 D terms of which each is rounded to a step of 2^-149 is
# off by 2^-150 sqrt(150 D) at most typically, 1e-2 of 1e-41 at D = 128; the
# large case loses nothing.
@pytest.mark.parametrize("den,bound", [(1e-41, 1e-2), (1.2e38, BOUND[torch.float32])])
@pytest.mark.parametrize("dtype,D", [(torch.float32, 16), (torch.float32, 32), (torch.float32, 64),
                                     (torch.float32, 128), (torch.bfloat16, 64), (torch.bfloat16, 128)])
def test_denominators_at_the_ends_of_the_range(dtype, D, den, bound):
    B, N, H = 1, 150, 3
    qkv = packed(B, N, H, D, torch.float32, seed=D)
    qkv[:, :, :2] *= (den / (24 * D)) ** 0.5
    qkv = qkv.to(dtype)
    want = exact(qkv, H, D, eps=0.0)
    got = linear_attention(qkv.to(DEV), H, D, eps=0.0)
    assert bool(torch.isfinite(got).all())
    assert rel(got.cpu(), want) <= bound
    assert rel(linear_attention(unaligned(qkv.to(DEV)), H, D, eps=0.0).cpu(), want) <= bound
