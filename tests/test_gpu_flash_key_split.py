"""The fused forward's key split: grids too short for 256-row blocks run 128-
or 64-row blocks whose waves share a query tile and add their parts of its keys
(64 bf16 heads at T = 512: two groups; a few heads: four).  Lengths around the
block and tile edges, windows, padded head dims, GQA, strided inputs, RoPE and
fp8, against the oracle."""
import math

import pytest
import torch

import smooth_attn
from oracle import eager
from smooth_attn import _lib, kernels

pytestmark = pytest.mark.gpu
DEV = "cuda"
TWO, FOUR = (2, 32, 8), (1, 4, 2)  # (B, Hq, Hkv) of grids that take 2 and 4 key groups at the lengths below
GROUPS = {TWO: 2, FOUR: 4}


def takes(heads, T, D, window, groups):
    """The launch takes the build with this many key groups (rows of D 16-bit elements, heads side by side)."""
    return _lib.load().sa_flash_fwd_key_split(*heads, T, D, window, 0, 2 * D * heads[2]) == groups


def rel_err(got, ref):
    got, ref = got.detach().double().cpu(), ref.detach().double().cpu()
    return float((got - ref).abs().max() / ref.abs().max().clamp(min=1e-30))


def qkv(heads, T, D, dtype, seed, bthd=False):
    B, Hq, Hkv = heads
    g = torch.Generator().manual_seed(seed)
    shape = (lambda H: (B, T, H, D)) if bthd else (lambda H: (B, H, T, D))
    out = [torch.randn(shape(H), generator=g).to(dtype) for H in (Hq, Hkv, Hkv)]
    return [t.transpose(1, 2) if bthd else t for t in out]


def check(q, k, v, window):
    o, rs = kernels._sp2norm_flash_fwd(q.to(DEV), k.to(DEV), v.to(DEV), 1.0 / math.sqrt(q.shape[-1]),
                                       q.shape[1] // k.shape[1], window)
    ref, ref_rs = eager.flash_attention_eager(q.double(), k.double(), v.double(), window_size=window,
                                              return_row_sums=True)
    assert bool(torch.isfinite(o).all())
    # weights and outputs rounded to 8 (11) bits once each; sums in fp32
    assert rel_err(o, ref) <= 1e-2
    assert rel_err(rs, ref_rs) <= 1e-5
    # the row sums of every row, first rows included (few keys)
    assert ((rs.cpu().double() - ref_rs).abs() <= 1e-5 * ref_rs).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("heads,T,D,window", [
    (FOUR, 256, 128, 0), (FOUR, 257, 128, 0), (FOUR, 319, 64, 0), (FOUR, 385, 32, 0), (FOUR, 511, 128, 1),
    (FOUR, 640, 128, 33), (FOUR, 640, 128, 192), (FOUR, 641, 96, 200), (FOUR, 1023, 128, 0), (FOUR, 1100, 40, 129), (FOUR, 2049, 64, 600),
    (TWO, 385, 128, 0), (TWO, 449, 64, 0), (TWO, 511, 32, 0), (TWO, 512, 128, 300), (TWO, 513, 72, 0),
    (TWO, 500, 128, 450)])
def test_key_split_matches_oracle(dtype, heads, T, D, window):
    assert takes(heads, T, D, window, GROUPS[heads])
    check(*qkv(heads, T, D, dtype, T + D), window)


@pytest.mark.parametrize("heads,T", [(FOUR, 300), (TWO, 500)])
def test_key_split_of_strided_inputs(heads, T):
    assert takes(heads, T, 128, 0, GROUPS[heads])
    check(*qkv(heads, T, 128, torch.bfloat16, 5, bthd=True), 0)


@pytest.mark.parametrize("heads,T,D", [(FOUR, 333, 128), (FOUR, 700, 64), (TWO, 511, 32)])
@pytest.mark.parametrize("v8", [True, False])
def test_key_split_fp8(heads, T, D, v8):
    assert takes(heads, T, D, 0, GROUPS[heads])
    q, k, v = qkv(heads, T, D, torch.bfloat16, T)
    (q8, qs), (k8, ks), (v8t, vs) = (eager.quantize_to_fp8(t) for t in (q, k, v))
    vv, vsc = (v8t, vs) if v8 else (v, 1.0)
    o, rs = kernels._sp2norm_fp8_flash_fwd(q8.to(DEV), k8.to(DEV), vv.to(DEV), float(qs), float(ks), float(vsc),
                                           1.0 / math.sqrt(D), q.shape[1] // k.shape[1])
    ref, ref_rs = eager.flash_attention_eager(q8.double() * float(qs), k8.double() * float(ks),
                                              vv.double() * float(vsc), return_row_sums=True)
    assert rel_err(o, ref) <= 1e-2
    assert rel_err(rs, ref_rs) <= 1e-5


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("heads,T,D", [(FOUR, 333, 128), (TWO, 511, 64)])
def test_key_split_rope(dtype, heads, T, D):
    assert takes(heads, T, D, 0, GROUPS[heads])
    q, k, v = qkv(heads, T, D, dtype, T + 1)
    cos, sin = smooth_attn.precompute_rope_cos_sin(D, T, device="cpu")
    o = smooth_attn.sp2norm_rope_flash_attention(q.to(DEV), k.to(DEV), v.to(DEV), cos.to(DEV), sin.to(DEV))
    ref = eager.rope_flash_attention_eager(q.double(), k.double(), v.double(), cos, sin, round_to=dtype)
    assert rel_err(o, ref) <= 1e-2


@pytest.mark.parametrize("bad", [math.inf, math.nan])
@pytest.mark.parametrize("heads,T,D,window", [
    (FOUR, 640, 128, 0), (FOUR, 577, 64, 0), (FOUR, 640, 128, 192), (FOUR, 641, 96, 200), (FOUR, 300, 32, 0),
    (TWO, 449, 64, 0), (TWO, 512, 128, 300)])
def test_non_finite_values_reach_the_same_rows_in_every_build(heads, T, D, window, bad):
    # 0 x Inf: a bad V row reaches rows that do not see its key where a wave
    # walks the key's tile.  The build without a key split (exact square
    # roots have no other) walks tiles of 64 keys.
    assert takes(heads, T, D, window, GROUPS[heads])
    q, k, v = (t.to(DEV) for t in qkv(heads, T, D, torch.bfloat16, 7))
    clean = smooth_attn.sp2norm_flash_attention(q, k, v, window_size=window)
    for key in (70, 127, 128, 191, 255, T - 40):
        vb = v.clone()
        vb[:, :, key, 3] = bad
        o = smooth_attn.sp2norm_flash_attention(q, k, vb, window_size=window)
        one = smooth_attn.sp2norm_flash_attention(q, k, vb, window_size=window, exact_math=True)
        hit = ~torch.isfinite(o)
        assert torch.equal(hit, ~torch.isfinite(one)), key
        assert torch.equal(o[~hit], clean[~hit])
        assert bool(hit[:, :, key, 3].all()) and not bool(hit[:, :, : key // 64 * 64].any())
