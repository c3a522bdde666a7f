"""RMSNorm's vectorised backward at the edges of its row shapes, against the
fp64 gradients of the exact formula and against the scalar kernel, which the
same call reaches when x is not 16-byte aligned.

x, dy and the weight are exact in fp64, so the fp64 gradients differ from the
kernel's by its roundings: n = tx(x inv) and g = tx(dy w) (half an ulp of tx
each, absent for fp32), fp32 sums (sqrt(n) 2^-24 relative, under 4e-6 here)
and one rounding of each result.  The relative 2-norm is therefore within the
sum of those half ulps.
"""

import pytest
import torch

from kernelforge_amd import _lib
from kernelforge_amd.rmsnorm.custom import rms_norm_module_forward

pytestmark = pytest.mark.gpu
DEV = "cuda"
F32, BF16, F16 = torch.float32, torch.bfloat16, torch.float16
HALF_ULP = {F32: 4e-6, BF16: 2.0 ** -8, F16: 2.0 ** -11}


def grads(x, w, dy):
    x, w = x.detach().requires_grad_(True), w.detach().requires_grad_(True)
    y = rms_norm_module_forward(x, w, 1e-6)
    return torch.autograd.grad(y, (x, w), dy.to(y.dtype))


def exact(x, w, dy):
    x, w = x.double().requires_grad_(True), w.double().requires_grad_(True)
    y = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * w
    return torch.autograd.grad(y, (x, w), dy.double())


def rel(a, b):
    return float((a.double() - b.double()).norm() / b.double().norm())


def offset_copy(t):
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=DEV)
    out = flat[1:].view(t.shape)
    out.copy_(t)
    return out


# One vector, the last and first width of each (vectors per lane, wavefronts
# per row) shape for 8-element vectors, and past the widest; rows that leave
# partly filled row slots, and more rows than blocks.
@pytest.mark.parametrize("dim", [8, 504, 512, 520, 1024, 1032, 2048, 2240, 4096, 4104, 8192, 8200, 16384, 16392])
@pytest.mark.parametrize("xdt,wdt", [(BF16, F32), (BF16, BF16), (F32, F32), (F16, F32), (F32, BF16)])
def test_row_shapes(dim, xdt, wdt):
    for rows in (1, 3, 37) + ((4100,) if dim in (512, 2240) else ()):
        g = torch.Generator().manual_seed(rows * 31 + dim)
        x = torch.randn(rows, dim, generator=g).to(xdt).to(DEV)
        w = (1 + 0.1 * torch.randn(dim, generator=g)).to(wdt).to(DEV)
        ydt = torch.promote_types(xdt, wdt)
        dy = torch.randn(rows, dim, generator=g).to(ydt).to(DEV)
        dx, dw = grads(x, w, dy)
        ex, ew = exact(x, w, dy)
        assert dx.dtype == xdt and dw.dtype == wdt
        assert rel(dx, ex) <= 2 * HALF_ULP[xdt], (rows, dim)
        assert rel(dw, ew) <= HALF_ULP[xdt] + HALF_ULP[wdt], (rows, dim)
        sx, sw = grads(offset_copy(x), w, dy)
        assert rel(dx, sx) <= 2 * HALF_ULP[xdt] and rel(dw, sw) <= HALF_ULP[wdt] + HALF_ULP[xdt]
        again = grads(x, w, dy)
        assert torch.equal(dx, again[0]) and torch.equal(dw, again[1])


def test_infinite_row_stays_in_its_row():
    """A row with an infinity or NaN leaves the other rows' dx as they are."""
    x = torch.randn(40, 1032, device=DEV).to(BF16)
    w = torch.ones(1032, device=DEV)
    dy = torch.randn(40, 1032, device=DEV)
    clean = grads(x, w, dy)[0]
    bad = x.clone()
    bad[5, 3] = float("inf")
    bad[17, 1031] = float("nan")
    dx = grads(bad, w, dy)[0]
    keep = torch.ones(40, dtype=torch.bool, device=DEV)
    keep[[5, 17]] = False
    assert torch.equal(dx[keep], clean[keep])
    assert bool(torch.isnan(dx[5]).any()) and bool(torch.isnan(dx[17]).all())


@pytest.mark.parametrize("dim", [8, 504, 1032, 2240, 4104])
def test_infinite_weight(dim):
    """An infinite weight makes its own column's dx infinite or NaN and the other
    columns' infinite, also where the row leaves vectors of a wavefront unused."""
    x = (1 + torch.rand(3, dim, device=DEV)).to(BF16)
    w = torch.ones(dim, device=DEV)
    w[0] = float("inf")
    dx, dw = grads(x, w, torch.ones(3, dim, device=DEV))
    assert bool(torch.isinf(dx[:, 1:]).all()) and bool(torch.isfinite(dw).all())


@pytest.mark.parametrize("rows", [0, 1])
def test_more_columns_than_one_reduction_launch_takes(rows):
    """2^28 columns at 16 threads each pass the 2^32 - 1 threads of one grid.
    Entries of +-1 have a mean square of 1 (their sums are exact), so dw is dy
    with x's signs; with no rows it is zero."""
    dim = 2 ** 28 + 40
    g = torch.Generator(DEV).manual_seed(rows)
    signs = torch.empty(rows, dim, device=DEV, dtype=BF16).bernoulli_(0.5, generator=g) * 2 - 1
    dy = torch.empty(rows, dim, device=DEV, dtype=BF16).normal_(generator=g)
    w = torch.ones(dim, device=DEV, dtype=BF16)
    dx, dw = torch.empty_like(signs), torch.full_like(w, float("nan"))
    lib = _lib.load()
    nbytes = lib.kf_rmsnorm_bwd_workspace_bytes(rows, dim)
    ws = torch.empty(nbytes, device=DEV, dtype=torch.uint8)
    _lib.check(lib.kf_rmsnorm_bwd(*map(_lib.ptr, (signs, w, dy, dx, dw, ws)), nbytes, rows, dim, 1e-6, _lib.KF_BF16,
                                  _lib.KF_BF16, _lib.stream_of(w)), "kf_rmsnorm_bwd")
    assert torch.equal(dw, (signs * dy)[0] if rows else torch.zeros_like(w))
