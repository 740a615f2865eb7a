"""Paged decode around the edges of its work plan: batches of up to 64 sequences
(planned by every wave) and more (planned by a kernel), empty contexts at the
ends and in runs, and segments cut into more than 16 and 64 partials."""
import pytest
import torch

import smooth_attn
from oracle import eager

pytestmark = pytest.mark.gpu
DEV = "cuda"
P = 16


def decode(lens, Hq, Hkv, D, seed):
    g = torch.Generator().manual_seed(seed)
    B = len(lens)
    width = max(max(lens) // P + 1, 1)
    total = B * width
    table = torch.randperm(total, generator=g).view(B, width).to(torch.int32)
    k = torch.randn(total, Hkv, P, D, generator=g).to(torch.bfloat16)
    v = torch.randn(total, Hkv, P, D, generator=g).to(torch.bfloat16)
    q = torch.randn(B, Hq, 1, D, generator=g).to(torch.bfloat16)
    ctx = torch.tensor(lens, dtype=torch.int32)
    out = smooth_attn.sp2norm_paged_attention(q.to(DEV), k.to(DEV), v.to(DEV), table.to(DEV), ctx.to(DEV),
                                              block_size=P)
    ref = eager.paged_decode_eager(q.double(), k.double(), v.double(), table, ctx)
    return out.cpu().double(), ref.double()


def check(lens, Hq, Hkv, D, seed):
    out, ref = decode(lens, Hq, Hkv, D, seed)
    # bf16 weights and outputs (2^-9 each of their values), fp32 sums
    assert float((out - ref).abs().max() / ref.abs().max()) <= 1e-2
    for b, n in enumerate(lens):
        if n == 0:
            assert int(out[b].count_nonzero()) == 0


@pytest.mark.parametrize("B", [1, 2, 63, 64, 65, 128, 130])
@pytest.mark.parametrize("D", [8, 64, 128])
def test_batch_sizes_around_the_wave_plan(B, D):
    lens = [(37 * b * b + 11 * b + 1) % 150 for b in range(B)]
    check(lens, 4, 2, D, B + D)


@pytest.mark.parametrize("B", [5, 64, 66])
def test_empty_contexts(B):
    lens = [0, 0] + [33 * (b % 3) for b in range(B - 4)] + [0, 0]
    lens[2] = 70
    check(lens, 2, 1, 64, B)
    out, _ = decode([0] * B, 2, 1, 64, 1)
    assert int(out.count_nonzero()) == 0


@pytest.mark.parametrize("ctx", [16 * 32 + 1, 17 * 32, 64 * 32, 65 * 32 + 5, 130 * 32])
def test_many_partials_per_segment(ctx):
    check([ctx], 2, 1, 128, ctx)
    check([ctx, 3, ctx - 40], 8, 2, 64, ctx)


@pytest.mark.parametrize("ctx", [32, 64, 96, 8 * 32, 9 * 32 + 1, 16 * 32, 17 * 32, 25 * 32, 70 * 32])
def test_many_partials_in_a_large_batch(ctx):
    # past 64 sequences the merge reads a segment's partials 2, 8 or 16 at a
    # time: one long segment of 1 to 70 partials among short ones
    check([5] * 40 + [ctx] + [0, 33] * 13, 4, 2, 64, ctx)
