"""kf_qk_norm_rope (q/k norm and rotary embedding in one pass) against the
kernels it stands for: the in-place row norm of q and of k, then
kf_rope_packed.  Same arithmetic in the same order: equal bit for bit."""

import pytest
import torch

from kernelforge_amd import _lib
from kernelforge_amd.rmsnorm.custom import rms_norm_rows_

pytestmark = pytest.mark.gpu
DEV = "cuda"


# One token; every row shape (wavefronts per row) at its first and last width
# for 2-byte types; odd token counts, which leave a block's second row empty;
# head dims that do and do not divide a wavefront's load.
@pytest.mark.parametrize("heads,dim", [(1, 8), (3, 8), (16, 32), (17, 32), (32, 32), (36, 32), (64, 32), (70, 32),
                                       (128, 32), (255, 16), (8, 128), (12, 24), (9, 72)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rope", [False, True])
def test_equals_separate_kernels(heads, dim, dtype, rope):
    C = heads * dim
    for B, N in ((1, 1), (2, 37)):
        g = torch.Generator().manual_seed(C + N)
        qkv = torch.randn(B, N, 3, C, generator=g).to(dtype).to(DEV)
        qw, kw = ((1 + 0.1 * torch.randn(C, generator=g)).to(dtype).to(DEV) for _ in range(2))
        angle = torch.rand(N, dim, generator=g).to(DEV) * 6
        cos, sin = angle.cos(), angle.sin()
        want = qkv.clone()
        rms_norm_rows_(want[:, :, 0], qw, 1e-5)
        rms_norm_rows_(want[:, :, 1], kw, 1e-5)
        lib = _lib.load()
        if rope:
            _lib.check(lib.kf_rope_packed(_lib.ptr(want), _lib.ptr(cos), _lib.ptr(sin), B, N, heads, dim,
                                          _lib.kf_dtype(dtype), _lib.stream_of(want)), "kf_rope_packed")
        got = qkv.clone()
        tables = (cos, sin) if rope else (None, None)
        _lib.check(lib.kf_qk_norm_rope(_lib.ptr(got), _lib.ptr(qw), _lib.ptr(kw), *map(_lib.ptr, tables), B, N, heads,
                                       dim, 1e-5, _lib.kf_dtype(dtype), _lib.stream_of(got)), "kf_qk_norm_rope")
        assert torch.equal(got, want)
        assert torch.equal(got[:, :, 2], qkv[:, :, 2])


def test_refuses_what_it_does_not_cover():
    lib = _lib.load()
    t = torch.zeros(1, 1, 3, 16384, device=DEV, dtype=torch.bfloat16)
    args = [_lib.ptr(t)] * 3 + [_lib.ptr(None)] * 2
    bf = _lib.kf_dtype(torch.bfloat16)
    assert lib.kf_qk_norm_rope(*args, 1, 1, 3, 4, 1e-5, bf, _lib.stream_of(t)) != 0      # 24-byte rows
    assert lib.kf_qk_norm_rope(*args, 1, 1, 512, 32, 1e-5, bf, _lib.stream_of(t)) != 0   # over 16 KiB
    assert lib.kf_qk_norm_rope(_lib.ptr(t[..., 1:]), *args[1:], 1, 1, 2, 32, 1e-5, bf, _lib.stream_of(t)) != 0


@pytest.mark.parametrize("rope", [False, True])
def test_more_rows_than_one_launch_takes(rope):
    """33.6 million tokens: 67.1 million rows of q and k, four to a workgroup of
    256 threads, pass the 2^32 - 1 threads of one grid inside a sequence."""
    B, N, D = 5, 6_711_000, 8
    assert 2 * B * N * 64 > 2 ** 32 - 1
    g = torch.Generator(DEV).manual_seed(3)
    got = torch.empty(B, N, 3, D, device=DEV, dtype=torch.bfloat16).normal_(generator=g)
    qw, kw = (torch.empty(D, device=DEV, dtype=torch.bfloat16).normal_(1, 0.1, generator=g) for _ in range(2))
    angle = torch.empty(N, D, device=DEV).uniform_(0, 6, generator=g)
    cos, sin = angle.cos(), angle.sin()
    want = got.clone()
    rms_norm_rows_(want[:, :, 0], qw, 1e-5)
    rms_norm_rows_(want[:, :, 1], kw, 1e-5)
    lib, bf, stream = _lib.load(), _lib.KF_BF16, _lib.stream_of(got)
    if rope:
        _lib.check(lib.kf_rope_packed(*map(_lib.ptr, (want, cos, sin)), B, N, 1, D, bf, stream), "kf_rope_packed")
    tables = (cos, sin) if rope else (None, None)
    _lib.check(lib.kf_qk_norm_rope(*map(_lib.ptr, (got, qw, kw, *tables)), B, N, 1, D, 1e-5, bf, stream),
               "kf_qk_norm_rope")
    assert torch.equal(got, want)
