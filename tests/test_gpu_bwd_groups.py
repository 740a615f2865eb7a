"""The attention backward's two-group blocks (8 waves, two for each 32-row tile,
merged in LDS): grids too short to fill the GPU take them, alone or with the
dK/dV split.  Lengths around tile and block edges, windows, GQA, padded head
dims, strided inputs; against float64 gradients."""
import ctypes
import math

import pytest
import torch

from oracle import eager
from smooth_attn import _lib, kernels

pytestmark = pytest.mark.gpu
DEV = "cuda"


def rel_err(got, ref):
    got, ref = got.detach().double().cpu(), ref.detach().double().cpu()
    return float((got - ref).abs().max() / ref.abs().max().clamp(min=1e-30))


def plan(B, Hq, Hkv, T, D, window, exact=0):
    """(dQ groups, dK/dV groups, splits) of the backward's launch."""
    lib, out = _lib.load(), (ctypes.c_int * 3)()
    ws = lib.sa_flash_bwd_workspace_size(B, Hq, Hkv, T, D, window, _lib.SA_BF16)
    assert lib.sa_flash_bwd_plan(B, Hq, Hkv, T, D, window, exact, ws, out) == 0
    return tuple(out)


def grads64(q, k, v, o, do, window):
    """dQ, dK, dV in float64 from the forward's rounded O (its rounding enters
    delta = dO . O), K and V expanded over the query heads and summed back."""
    G, Hkv = q.shape[1] // k.shape[1], k.shape[1]
    B, _, T, D = q.shape
    rq, rk, rv = eager.flash_attention_bwd(q.double(), k.double().repeat_interleave(G, 1),
                                           v.double().repeat_interleave(G, 1), o.cpu().double(), do.double(),
                                           scale=1.0 / math.sqrt(D), window_size=window)
    return rq, rk.reshape(B, Hkv, G, T, D).sum(2), rv.reshape(B, Hkv, G, T, D).sum(2)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,Hq,Hkv,T,D,window,groups", [
    (2, 8, 8, 512, 128, 0, (2, 2)), (2, 8, 8, 513, 64, 0, (2, 2)), (1, 8, 8, 575, 32, 0, (2, 2)),
    (2, 4, 4, 640, 96, 0, (2, 2)), (1, 8, 8, 700, 40, 0, (2, 1)), (1, 8, 8, 575, 40, 0, (2, 2)),
    (1, 16, 4, 577, 64, 0, (2, 2)), (1, 8, 2, 1025, 128, 0, (2, 2)), (1, 8, 8, 900, 128, 130, (1, 2)),
    (1, 8, 8, 900, 128, 400, (2, 2)), (1, 8, 2, 800, 64, 65, (1, 2)), (1, 4, 4, 1100, 128, 1, (1, 1)),
    (1, 16, 2, 600, 80, 333, (2, 2))])
def test_groups_match_float64(dtype, B, Hq, Hkv, T, D, window, groups):
    # groups of the dQ and the dK/dV blocks: short windows leave them little to share
    assert plan(B, Hq, Hkv, T, D, window)[:2] == groups
    g = torch.Generator().manual_seed(T + D)
    mk = lambda H: torch.randn(B, T, H, D, generator=g).to(dtype).transpose(1, 2)  # rows of all heads side by side
    q, k, v, do = mk(Hq), mk(Hkv), mk(Hkv), mk(Hq)
    scale = 1.0 / math.sqrt(D)
    dev = [t.to(DEV) for t in (q, k, v, do)]
    o, rs = kernels._sp2norm_flash_fwd(*dev[:3], scale, Hq // Hkv, window)
    got = kernels._sp2norm_flash_bwd(*dev[:3], o, dev[3], rs, scale, Hq // Hkv, window)
    again = kernels._sp2norm_flash_bwd(*dev[:3], o, dev[3], rs, scale, Hq // Hkv, window)
    for name, x, y, ref in zip(("dq", "dk", "dv"), got, again, grads64(q, k, v, o, do, window)):
        assert torch.equal(x, y), name  # sums run in a fixed order
        assert bool(torch.isfinite(x).all())
        # P, dS and the results rounded to 8 (11) bits, sums in fp32; with one
        # key per query dQ and dK cancel to rounding noise, so never below 1e-2
        err = float((x.double().cpu() - ref).abs().max() / max(float(ref.abs().max()), 1.0 if window == 1 else 1e-2))
        assert err <= 1e-2, (name, err)


def test_exact_square_roots_keep_one_group():
    # (no two-group build): same gradients as the fast build within rounding
    assert plan(1, 8, 8, 513, 64, 0)[:2] == (2, 2) and plan(1, 8, 8, 513, 64, 0, 1)[:2] == (1, 1)
    g = torch.Generator().manual_seed(1)
    q, k, v, do = (torch.randn(1, 8, 513, 64, generator=g).to(torch.bfloat16).to(DEV) for _ in range(4))
    o, rs = kernels._sp2norm_flash_fwd(q, k, v, 0.125, 1, 0)
    a = kernels._sp2norm_flash_bwd(q, k, v, o, do, rs, 0.125, 1, 0)
    b = kernels._sp2norm_flash_bwd(q, k, v, o, do, rs, 0.125, 1, 0, use_fast_sqrt=False)
    for x, y in zip(a, b):
        assert rel_err(x, y) <= 1e-2
