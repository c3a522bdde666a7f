"""The projection GEMM's small output tiles (64x64, 128x64, 128x128): every
tile adds an output's products in the same K order, so each result equals the
256-row tile's bit for bit; integer inputs (exact in fp32) also equal the fp64
product rounded once."""

import pytest
import torch

from kernelforge_amd import _lib
from kernelforge_amd.SANA_LinearAttention.projection import linear

pytestmark = pytest.mark.gpu
DEV = "cuda"


def run(x, w, b, tile):
    m, k = x.shape
    n = w.shape[0]
    y = torch.full((m, n), float("nan"), device=DEV, dtype=x.dtype)
    rc = _lib.load().kfm_proj_gemm_tile(_lib.ptr(x), _lib.ptr(w), _lib.ptr(b), _lib.ptr(y), m, n, k, k, n,
                                        _lib.KF_WEIGHT_NK, _lib.kf_dtype(x.dtype), tile, _lib.stream_of(x))
    _lib.check(rc, "kfm_proj_gemm_tile")
    return y


# One row and column chunk; tile edges +-1 row and +-8 columns; a K of one
# chunk, of fewer stages than a tile keeps in flight, and with a partial stage.
@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (63, 64, 64), (65, 72, 72), (127, 56, 128), (129, 136, 200),
                                   (300, 264, 1160), (577, 704, 704)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bias", [False, True])
def test_tiles_agree(M, N, K, dtype, bias):
    g = torch.Generator().manual_seed(M + N)
    x, w, b = (torch.randn(s, generator=g).to(dtype).to(DEV) for s in ((M, K), (N, K), (N,)))
    b = b if bias else None
    want = run(x, w, b, 128)
    for tile in (1, 2, 3):
        assert torch.equal(run(x, w, b, tile), want), tile
    assert torch.equal(linear(x, w, b), want)
    xi, wi, bi = (torch.randint(-3, 4, s, generator=g).to(dtype) for s in ((M, K), (N, K), (N,)))
    exact = (xi.double() @ wi.double().T + (bi.double() if bias else 0)).to(dtype)
    for tile in (1, 2, 3):
        assert torch.equal(run(xi.to(DEV), wi.to(DEV), bi.to(DEV) if bias else None, tile).cpu(), exact), tile


def test_more_rows_than_a_small_tile_grid_takes():
    """537 million rows of 8 columns: 64-row tiles of 512 threads pass the
    2^32 - 1 threads of one grid, the 256-row tiles do not."""
    M, K, N = 2 ** 29 + 100, 8, 8
    g = torch.Generator(DEV).manual_seed(1)
    x = torch.empty(M, K, device=DEV, dtype=torch.bfloat16).random_(-3, 4, generator=g)
    w = torch.empty(N, K, device=DEV, dtype=torch.bfloat16).random_(-3, 4, generator=g)
    y = linear(x, w)
    for r0 in (0, M // 2, M - 5000):
        rows = x[r0:r0 + 5000].cpu().double()
        assert torch.equal(y[r0:r0 + 5000].cpu(), (rows @ w.cpu().double().T).to(torch.bfloat16))
