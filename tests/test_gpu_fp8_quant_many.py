"""Per-tensor fp8 quantisation of several tensors in one pair of launches, and
its quotient: codes and scales against the CPU's true fp32 division."""
import pytest
import torch

from oracle import eager
from smooth_attn import kernels

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _check(x8, scale, x):
    # whole results: a scale is one fp32 division, a code one fp32 division
    # and one rounding, so both are equal bit for bit
    ref8, ref_scale = eager.quantize_to_fp8(x.cpu())
    assert float(scale) == float(ref_scale)
    assert torch.equal(x8.view(torch.uint8).cpu(), ref8.view(torch.uint8))


# a lone element, remainders below a 16-byte step, one and several blocks, more
# than the amax pass's blocks hold at one load a lane; sizes far apart, whose
# blocks are dealt out unevenly
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("sizes", [(1,), (7, 1, 3), (8192, 8191, 8193), (9_000_011, 5, 70_001), (1 << 21, 1 << 19, 1 << 19),
                                   (100, 200, 300, 400)])
def test_many_matches_one_by_one(dtype, sizes):
    g = torch.Generator().manual_seed(sum(sizes))
    xs = [(torch.randn(n, generator=g) * 10.0 ** (i - 1)).to(dtype) for i, n in enumerate(sizes)]
    for (x8, scale), x in zip(kernels._quantize_many_to_fp8_device(*[x.to(DEV) for x in xs]), xs):
        _check(x8, scale, x)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_many_with_unaligned_and_empty(dtype):
    g = torch.Generator().manual_seed(3)
    base = (torch.randn(70_001, generator=g) * 5).to(dtype).to(DEV)
    empty = torch.empty(0, 4, dtype=dtype, device=DEV)
    (a8, a_s), (b8, b_s), (e8, e_s) = kernels._quantize_many_to_fp8_device(base[1:], base[:-1], empty)
    _check(a8, a_s, base[1:])
    _check(b8, b_s, base[:-1])
    assert e8.shape == (0, 4) and float(e_s) == pytest.approx(1e-12)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("amax", [2.0 ** -24, 3e-5, 0.3, 1.0, 447.0, 448.0, 449.0, 61440.0])
def test_quotient_over_every_value(dtype, amax):
    # every finite value of the type up to the largest, zeros of both signs
    # and denormals included, under scales of all sizes
    bits = torch.arange(1 << 16, dtype=torch.int32).to(torch.int16)
    x = bits.view(dtype)
    x = x[torch.isfinite(x.float()) & (x.float().abs() <= amax)]
    (x8, scale), = kernels._quantize_many_to_fp8_device(x.to(DEV))
    _check(x8, scale, x)


def test_infinite_scale():
    # finite values divide to zeros of their own sign, infinite ones to NaN,
    # which the clamp takes to its lower end
    x = torch.tensor([float("inf"), 1.0, -1.0, 0.0, -0.0, float("-inf")], dtype=torch.bfloat16, device=DEV)
    many = kernels._quantize_many_to_fp8_device(x, x)
    wide = kernels._quantize_to_fp8_device(x.float())  # fp32 divides
    for x8, scale in many:
        assert float(scale) == float("inf")
        assert torch.equal(x8.view(torch.uint8), wide[0].view(torch.uint8))


def _one_word(x, dirty):
    """sa_fp8_quantize: one word of workspace, whatever it holds."""
    from smooth_attn import _lib

    lib = _lib.load()
    x8 = torch.full((max(x.numel(), 1),), 0x55, dtype=torch.uint8, device=DEV)
    ws = torch.tensor([dirty], dtype=torch.int32, device=DEV)
    scale = torch.zeros(1, dtype=torch.float32, device=DEV)
    st = lib.sa_fp8_quantize(x.data_ptr(), x8.data_ptr(), x.numel(), kernels._DTYPE_CODE[x.dtype], ws.data_ptr(),
                             scale.data_ptr(), kernels._stream(x8))
    assert st == 0
    return x8, scale


# a lone element, remainders, one block, the most blocks that meet in the word
# (256, one per CU) and several loads of each; an address between 16-byte ones;
# nothing at all; a workspace that holds zero, a large float's bits, NaN bits
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("n,offset", [(0, 0), (1, 0), (7, 0), (8192, 0), (8193, 1), (70_001, 1), (1 << 21, 0), (9_000_011, 0)])
def test_one_word_workspace_matches_many(dtype, n, offset):
    g = torch.Generator(device=DEV).manual_seed(n)
    x = (torch.randn(n + offset, generator=g, device=DEV) * 3).to(dtype)[offset:]
    (want8, want), = kernels._quantize_many_to_fp8_device(x)
    for dirty in (0, 0x7F000000, -1):
        x8, scale = _one_word(x, dirty)
        assert torch.equal(scale, want.reshape(1))
        assert torch.equal(x8[:n], want8.view(torch.uint8).reshape(-1))
        assert n > 0 or int(x8[0]) == 0x55  # nothing written


@pytest.mark.parametrize("sizes", [((81 << 20) + 5,), (84 << 20, 1000, 7)])
def test_inputs_past_the_caches(sizes):
    # over 320 MiB of fp32 the passes stream: codes and scales of each tensor
    # as alone, where it is short, and as one division per element says
    g = torch.Generator(device=DEV).manual_seed(1)
    xs = [torch.randn(n, generator=g, device=DEV) * 2 for n in sizes]
    for (x8, scale), x in zip(kernels._quantize_many_to_fp8_device(*xs), xs):
        assert float(scale) == float(x.abs().max().cpu() / 448.0)  # one fp32 division, on the CPU
        for part in (x[:4096], x[-4096:], x[x.numel() // 2:][:4096]):
            i = (part.data_ptr() - x.data_ptr()) // 4
            want = (part.cpu() / scale.cpu()).clamp(-448, 448).to(torch.float8_e4m3fn)
            assert torch.equal(x8[i:i + part.numel()].cpu().view(torch.uint8), want.view(torch.uint8))
