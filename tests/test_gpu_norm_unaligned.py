"""Normalisation rows that are not 16-byte aligned, or whose length is no
multiple of a 16-byte load: lengths around the chunk boundaries of the one-wave
and split-row kernels, wider row strides, bases off by one element, and a
gradient of the other type.  Rows lie in a larger buffer whose gaps must stay
untouched."""
import pytest
import torch

from oracle import eager
from smooth_attn import kernels
from smooth_attn.kernels import FamilyConfig

pytestmark = pytest.mark.gpu
DEV = "cuda"
MARK = -7.0  # in every element between the rows (exact in each type)


def _rows(data, stride, offset):
    """data [n, L] as rows `stride` apart, `offset` elements into a marked buffer."""
    n, L = data.shape
    buf = torch.full((offset + n * stride + 64,), MARK, dtype=data.dtype, device=DEV)
    view = buf[offset:offset + n * stride].view(n, stride)[:, :L]
    view.copy_(data)
    return buf, view


def _gaps_untouched(buf, n, L, stride, offset):
    rest = buf.clone()
    rest[offset:offset + n * stride].view(n, stride)[:, :L] = MARK
    return bool((rest == MARK).all())


# 16-bit: one rounding of the result (2^-9 of it) plus fp32 arithmetic; fp32:
# sums of up to 8192 terms by lanes and a tree, under 100 roundings of 2^-24.
def _tol(dtype):
    return 2.0 ** -8 if dtype != torch.float32 else 6e-6


def _cond(a, power):
    """Relative fp32 error of (a + sqrt(a^2 + 4))^power: the sum cancels where
    a < 0, and its terms carry up to 4 roundings of 2^-24."""
    r = torch.sqrt(a * a + 4.0)
    return power * 2.0 ** -22 * (a.abs() + r) / (a + r)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("L,extra,offset", [(255, 0, 0), (256, 1, 0), (257, 0, 0), (319, 0, 0), (321, 0, 0), (505, 0, 1), (511, 0, 0), (513, 0, 0),
                                            (520, 1, 0), (1023, 0, 0), (1025, 3, 1), (2049, 0, 0), (4095, 0, 0),
                                            (4097, 0, 1), (8191, 0, 0), (8192, 1, 1)])
@pytest.mark.parametrize("causal", [True, False])
def test_rows_at_any_address(dtype, L, extra, offset, causal):
    # causal rows take their position from row % L: the rows below are 0 .. n - 1
    gen = torch.Generator().manual_seed(L + 7 * extra + offset)
    n = L if causal and L <= 1100 else 9
    stride = L + extra
    fam = FamilyConfig()
    x = torch.randn(n, L, generator=gen).to(dtype).to(DEV)
    g = torch.randn(n, L, generator=gen).to(dtype).to(DEV)
    _, xv = _rows(x, stride, offset)
    ybuf, yv = _rows(torch.zeros_like(x), stride, offset)
    kernels._norm_fwd_2d(xv, yv, fam, causal)
    xd, gd = x.cpu().double(), g.cpu().double()
    w = eager.family_weights(xd, fam.alpha, fam.theta, fam.power)
    a = fam.alpha * (xd - fam.theta)
    if causal:
        w = torch.tril(w)
    S = w.sum(-1, keepdim=True) + 1e-12
    y = w / S
    slope, T = fam.alpha * fam.power * y / torch.sqrt(a * a + 4.0), (gd * y).sum(-1, keepdim=True)
    dx = slope * (gd - T)
    # dy - T cancels (in row 0 wholly): its fp32 terms carry the error of the sums
    near = 6e-6 * slope * (gd.abs() + (gd.abs() * y).sum(-1, keepdim=True))
    cond = _cond(a, fam.power)
    tol = _tol(dtype)
    tiny = 2.0 ** -24 if dtype == torch.float16 else 0.0  # fp16 subnormal spacing
    assert ((yv.cpu().double() - y).abs() <= (tol + cond) * y + tiny).all()
    assert not causal or int(yv[torch.triu(torch.ones(n, L, dtype=torch.bool, device=DEV), 1)].count_nonzero()) == 0
    assert _gaps_untouched(ybuf, n, L, stride, offset)
    for gdt in {dtype, torch.float32}:
        _, gv = _rows(g.to(gdt), stride, offset)
        dbuf, dv = _rows(torch.zeros_like(x), stride, offset)
        kernels._norm_bwd_2d(xv, gv, dv, fam, causal)
        assert ((dv.cpu().double() - dx).abs() <= (tol + cond) * dx.abs() + 2 * near + tiny).all()
        assert _gaps_untouched(dbuf, n, L, stride, offset)


@pytest.mark.parametrize("power", [1, 3])
def test_other_powers(power):
    fam = FamilyConfig(alpha=1.5, theta=0.25, power=power)
    x = torch.randn(2, 333, 333, generator=torch.Generator().manual_seed(3)).to(DEV)
    y = torch.empty_like(x)
    kernels._norm_fwd_2d(x.view(-1, 333), y.view(-1, 333), fam, True)
    ref = eager.softplus_norm_causal_eager(x.cpu().double(), fam.alpha, fam.theta, power)
    cond = _cond(fam.alpha * (x.cpu().double() - fam.theta), power)
    assert ((y.cpu().double() - ref).abs() <= (6e-6 + cond) * ref).all()
