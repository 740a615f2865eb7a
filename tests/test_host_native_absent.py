"""Calls refused by the device checks never load the native call path: the
outcome is the same whichever call of the process comes first, and where the
libraries are not built."""
import pytest
import torch

import smooth_attn
from smooth_attn import _lib


def _calls():
    q = torch.zeros(1, 4, 16, 32)
    k = torch.zeros(1, 2, 16, 32)
    x = torch.zeros(8, 8)
    cache = torch.zeros(4, 2, 16, 32)
    table, lens = torch.zeros(1, 4, dtype=torch.int32), torch.ones(1, dtype=torch.int32)
    return {
        "flash": lambda: smooth_attn.sp2norm_flash_attention(q, k, k),
        "paged": lambda: smooth_attn.sp2norm_paged_attention(q[:, :, :1], cache, cache, table, lens),
        "append": lambda: smooth_attn.sp2norm_paged_kv_append(cache, cache, k[:, :, :2], k[:, :, :2], table, lens),
        "causal norm": lambda: smooth_attn.softplus_norm_causal(x),
        "causal norm out": lambda: smooth_attn.softplus_norm_causal_triton_out(x.clone(), x),
        "row-wise out": lambda: smooth_attn.softplus_norm_triton_out(x.clone(), x),
    }


@pytest.mark.parametrize("name", sorted(_calls()))
def test_host_tensors_are_refused_without_the_libraries(name, monkeypatch):
    def fail():
        raise AssertionError("the libraries were loaded before the device check")

    monkeypatch.setattr(_lib, "load", fail)
    monkeypatch.setattr(_lib, "_host", None)
    monkeypatch.setattr(torch.cuda, "is_initialized", lambda: False)
    with pytest.raises(ValueError, match="must be a CUDA tensor"):
        _calls()[name]()
