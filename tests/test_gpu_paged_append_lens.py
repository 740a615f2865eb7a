"""The append's lengths, written by the same launch as the rows: whole numbers,
so equal to torch's addition."""
import ctypes

import pytest
import torch

import smooth_attn
from oracle import paging
from smooth_attn import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# fewer lengths than threads, as many, and more than the whole launch (B H n_new
# D / 8 chunks in blocks of 256): one row of one chunk leaves 256 threads
@pytest.mark.parametrize("count", [1, 255, 256, 257, 5000])
@pytest.mark.parametrize("n_new", [1, 3])
def test_lengths_beyond_the_batch(count, n_new):
    P, D = 16, 8
    g = torch.Generator().manual_seed(count)
    k = torch.randn(1, 1, 40, D, generator=g).bfloat16()
    kc, vc, table, _ = paging.build_paged_cache(k, k, P, generator=g)
    lens = torch.randint(-5, 1 << 30, (count,), generator=g, dtype=torch.int32)
    lens[0] = 37 - n_new
    new = torch.randn(1, 1, n_new, D, generator=g).bfloat16()
    ref_k, ref_v = paging.append_kv(kc, vc, new, -new, table, lens[:1])
    kd, vd, ld = kc.to(DEV), vc.to(DEV), lens.to(DEV)
    out = smooth_attn.sp2norm_paged_kv_append(kd, vd, new.to(DEV), -new.to(DEV), table.to(DEV), ld, block_size=P)
    assert out.dtype == torch.int32 and torch.equal(out.cpu(), lens + n_new)
    assert torch.equal(ld.cpu(), lens) and torch.equal(kd.cpu(), ref_k) and torch.equal(vd.cpu(), ref_v)


@pytest.mark.parametrize("B,n_new,pages", [(0, 2, 4), (3, 0, 4), (3, 2, 0)])
def test_lengths_without_rows(B, n_new, pages):
    # nothing to write to the caches: the lengths are written all the same
    lens = torch.arange(7, dtype=torch.int32, device=DEV)
    out = torch.full_like(lens, -1)
    s = (ctypes.c_int64 * 4)(0, 0, 0, 1)
    st = _lib.load().sa_paged_kv_append_lens(None, None, None, None, None, lens.data_ptr(), out.data_ptr(), 7, B, 2,
                                             n_new, 64, 16, pages, pages, s, s, s, pages, _lib.SA_BF16,
                                             torch.cuda.current_stream().cuda_stream)
    assert st == 0
    assert torch.equal(out, lens + n_new)
