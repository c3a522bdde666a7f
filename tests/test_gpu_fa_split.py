"""The split forward (fa_split_kernel, fa_combine_kernel): every key split and
row packing against the one-workgroup-per-tile kernel and the fp64 oracle.

Both kernels form P in 16 bits relative to a running row reference and sum in
fp32, so each is within the rounding of P (2^-8 relative for bf16, 2^-11 for
fp16, on every term) plus half an ulp of the result of the exact value; the
bounds are the suite's 3e-2 / 3e-3.  The LSE is an fp32 sum: 1e-3.
"""

import pytest
import torch

from kernelforge_amd import _lib
from kernelforge_amd.flash_attention_jvp import flash_attention, flash_attention_fwd_jvp
from oracle import fa as orc

pytestmark = pytest.mark.gpu
DEV = "cuda"
BOUNDS = {torch.float16: dict(atol=3e-3, rtol=1e-2), torch.bfloat16: dict(atol=3e-2, rtol=3e-2)}


def tensors(B, Nq, Nk, Hq, Hkv, D, dtype, seed=5):
    g = torch.Generator().manual_seed(seed)
    return tuple(torch.randn(s, generator=g).to(dtype).to(DEV)
                 for s in ((B, Nq, Hq, D), (B, Nk, Hkv, D), (B, Nk, Hkv, D)))


def forced(q, k, v, causal, splits, pack, tangents=(None, None, None), jvp=False, cached=None):
    B, Nq, Hq, D = q.shape
    Nk, Hkv = k.shape[1:3]
    out, lse = cached or (torch.full_like(q, float("nan")), torch.full((B, Hq, Nq), float("nan"), device=DEV))
    to = torch.full_like(q, float("nan")) if jvp else None
    ws = torch.full((max(splits, 1) * B * Hq * Nq * (2 * D + 4),), float("nan"), device=DEV)
    rc = _lib.load().kfm_fa_fwd_split(_lib.ptr(q), _lib.ptr(k), _lib.ptr(v), *map(_lib.ptr, tangents),
                                      _lib.ptr(out), _lib.ptr(lse), _lib.ptr(to), _lib.ptr(ws), ws.numel() * 4, B, Nq, Nk, Hq, Hkv, D, D ** -0.5, int(causal),
                                      _lib.kf_dtype(q.dtype), splits, int(pack), int(cached is not None),
                                      _lib.stream_of(q))
    _lib.check(rc, "kfm_fa_fwd_split")
    return (out, lse, to) if jvp else (out, lse)


# One row, tile edges of 128 rows and 64 (D > 128: 32) keys, packed groups that
# straddle 16-row blocks and 128-row tiles, more queries than keys (causal rows
# without a key), splits without a tile of their own.
CASES = [(1, 1, 1, 2, 2, 64, False), (2, 4, 700, 8, 2, 128, True), (1, 33, 129, 6, 2, 72, True),
         (1, 130, 65, 3, 3, 32, False), (2, 129, 515, 4, 1, 64, True), (1, 71, 19, 4, 1, 96, True),
         (1, 70, 200, 4, 2, 256, True), (1, 5, 333, 16, 1, 136, False)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", CASES)
def test_every_split(case, dtype):
    causal = case[-1]
    q, k, v = tensors(*case[:-1], dtype)
    tangents = tensors(*case[:-1], dtype, seed=6)
    want, want_t = orc.attention_jvp(*(t.cpu().double() for t in (q, k, v, *tangents)), causal=causal)
    lse_want = orc.attention_lse(q.cpu().double(), k.cpu().double(), causal=causal)
    for splits, pack in ((0, 0), (1, 0), (1, 1), (2, 0), (3, 1), (7, 1), (64, 0)):
        out, lse = forced(q, k, v, causal, splits, pack)
        torch.testing.assert_close(out.cpu().double(), want, **BOUNDS[dtype])
        torch.testing.assert_close(lse.cpu().double(), lse_want, atol=1e-3, rtol=1e-4)
        again = forced(q, k, v, causal, splits, pack)
        assert torch.equal(out, again[0]) and torch.equal(lse, again[1])
        # The fused forward + JVP over the same split: the same LSE sum.
        o2, lse2, to = forced(q, k, v, causal, splits, pack, tangents, jvp=True)
        assert torch.equal(lse2, lse)
        torch.testing.assert_close(o2.cpu().double(), want, **BOUNDS[dtype])
        torch.testing.assert_close(to.cpu().double(), want_t, **BOUNDS[dtype])
    # The JVP from cached results: one range is fa_kernel's own sum.
    cached = forced(q, k, v, causal, 0, 0)
    for splits in (0, 1, 2, 7, 64):
        to = forced(q, k, v, causal, splits, 0, tangents, True, cached)[2]
        torch.testing.assert_close(to.cpu().double(), want_t, **BOUNDS[dtype])
        if splits == 0:
            plain = to
        if splits == 1:
            assert torch.equal(to, plain)
    # Absent tangents are zeros.
    zero = torch.zeros_like(tangents[1])
    some = forced(q, k, v, causal, 3, 1, (tangents[0], None, tangents[2]), jvp=True)
    full = forced(q, k, v, causal, 3, 1, (tangents[0], zero, tangents[2]), jvp=True)
    torch.testing.assert_close(some[2], full[2], **BOUNDS[dtype])
    out, lse = flash_attention(q, k, v, causal=causal, return_lse=True)
    torch.testing.assert_close(out.cpu().double(), want, **BOUNDS[dtype])
    torch.testing.assert_close(lse.cpu().double(), lse_want, atol=1e-3, rtol=1e-4)


@pytest.mark.parametrize("splits,pack", [(1, 0), (4, 1)])
def test_growing_scores_rescale(splits, pack):
    """Scores that grow far past the first keys' maximum (the fixed-reference
    kernel's fixup case) stay finite and exact."""
    q, k, v = tensors(1, 40, 1000, 4, 2, 64, torch.bfloat16)
    k = (k * torch.linspace(0.1, 30, 1000, device=DEV)[None, :, None, None]).to(torch.bfloat16)
    out, lse = forced(q, k, v, False, splits, pack)
    want, _ = orc.attention_jvp(*(t.cpu().double() for t in (q, k, v)), *(torch.zeros_like(t).cpu().double()
                                                                         for t in (q, k, v)))
    torch.testing.assert_close(out.cpu().double(), want, **BOUNDS[torch.bfloat16])
    torch.testing.assert_close(lse.cpu().double(), orc.attention_lse(q.cpu().double(), k.cpu().double()),
                               atol=1e-3, rtol=1e-4)


@pytest.mark.parametrize("splits", [0, 3])
def test_jvp_peaked_tiles_recompute_the_output(splits):
    """Tiles past the cached-O bound (a strongly peaked softmax) are redone with
    O recomputed: the result does not depend on the cached out there, and does
    on tiles under the bound."""
    q, k, v = tensors(1, 256, 300, 2, 2, 64, torch.bfloat16)
    tangents = tensors(1, 256, 300, 2, 2, 64, torch.bfloat16, seed=6)
    q = q.clone()
    q[:, 128:] *= 16  # the second 128-row tile is peaked
    out, lse = forced(q, k, v, False, 0, 0)
    plain = forced(q, k, v, False, splits, 0, tangents, True, (out, lse))[2]
    moved = forced(q, k, v, False, splits, 0, tangents, True, (out + 0.25, lse))[2]
    assert torch.equal(plain[:, 128:], moved[:, 128:])
    assert not torch.equal(plain[:, :128], moved[:, :128])
    _, want = orc.attention_jvp(*(t.cpu().double() for t in (q, k, v, *tangents)))
    torch.testing.assert_close(plain.cpu().double(), want, **BOUNDS[torch.bfloat16])


def test_nan_key_stays_in_its_head():
    q, k, v = tensors(1, 8, 600, 4, 2, 64, torch.bfloat16)
    clean = forced(q, k, v, False, 4, 1)[0]
    k[0, 300, 1, 5] = float("nan")
    out = forced(q, k, v, False, 4, 1)[0]
    assert torch.equal(out[:, :, :2], clean[:, :, :2])
    assert bool(torch.isnan(out[:, :, 2:]).all()) == bool(torch.isnan(forced(q, k, v, False, 0, 0)[0][:, :, 2:]).all())


# Scores that rise far past the first keys' maximum, without overflow (2^128 over
# it in bf16, 2^16 in fp16).
@pytest.mark.parametrize("dtype,growth,ref", [(torch.bfloat16, 10, 128), (torch.float16, 1.5, 16)])
@pytest.mark.parametrize("shape", [(1, 333, 333, 16, 16, 64), (1, 700, 700, 16, 16, 128)])
def test_one_range_lse_of_both_modes(shape, dtype, growth, ref):
    """With one key range the forward rescales and the fused mode keeps its first
    reference.  Exponents of up to ``ref`` log2 units from it carry half an ulp of
    ref, which the sum, its log2 and the product with ln 2 each add once more at
    most (scores here stay under 128 log2 units): 4 * 2^-17 * ln 2 in the worse mode,
    twice that between the two."""
    q, k, v = tensors(*shape, dtype)
    k = (k * torch.linspace(0.1, growth, shape[2], device=DEV)[None, :, None, None]).to(dtype)
    tangents = tensors(*shape, dtype, seed=6)
    out, lse = flash_attention(q, k, v, return_lse=True)
    out2, lse2, tangent = flash_attention_fwd_jvp(q, k, v, *tangents)
    want, want_t = orc.attention_jvp(*(t.cpu().double() for t in (q, k, v, *tangents)))
    lse_want = orc.attention_lse(q.cpu().double(), k.cpu().double())
    scores = torch.einsum("bqhd,bkhd->bhqk", q.cpu().double(), k.cpu().double()) * shape[-1] ** -0.5 * 1.4427
    rise = (scores.amax(-1) - scores[..., :32].amax(-1)).amax()
    assert 8 < float(rise) < ref and float(scores.abs().max()) < 128
    bound = 8 * 2.0 ** -17 * 0.6932
    for got, exact in ((lse, lse_want), (lse2, lse_want), (lse, lse2)):
        torch.testing.assert_close(got.cpu().double(), exact.cpu().double(), atol=bound, rtol=0)
    for got, exact in ((out, want), (out2, want), (tangent, want_t)):
        scale = max(1.0, float(exact.abs().max()))
        torch.testing.assert_close(got.cpu().double() / scale, exact / scale, **BOUNDS[dtype])
