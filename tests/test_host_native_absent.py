"""Calls refused by the device checks never load the native call path: the
outcome is the same whichever call of the process comes first, and where the
libraries are not built.  Without the extension every call takes the Python
path."""
import warnings

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


@pytest.mark.parametrize("name", sorted(_calls()))
def test_host_tensors_are_refused_where_the_library_is_not_built(name, monkeypatch, tmp_path):
    monkeypatch.setattr(_lib, "LIB_PATH", tmp_path / "none.so")
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "_host", None)
    monkeypatch.setattr(torch.cuda, "is_initialized", lambda: True)
    with pytest.raises(ValueError, match="must be a CUDA tensor"):
        _calls()[name]()


def _no_file(path):
    pass


def _no_library(path):
    path.write_bytes(b"not a library")


@pytest.mark.parametrize("make", [_no_file, _no_library])
def test_without_the_extension_the_python_path_takes_every_call(make, monkeypatch, tmp_path):
    make(tmp_path / "_host.so")
    monkeypatch.setattr(_lib, "_HOST_PATH", tmp_path / "_host.so")
    monkeypatch.setattr(_lib, "_host", None)
    monkeypatch.setattr(torch.cuda, "is_initialized", lambda: True)
    with pytest.warns(RuntimeWarning, match="native call path not available"):
        assert smooth_attn.kernels._native().flash() is None
    with warnings.catch_warnings():  # said once
        warnings.simplefilter("error")
        assert smooth_attn.kernels._native().norm_out() is None
        for name, call in _calls().items():
            with pytest.raises(ValueError, match="must be a CUDA tensor"):
                call()


def test_an_extension_of_another_torch_is_not_used(monkeypatch):
    monkeypatch.setattr(torch, "__version__", "1.0.0+rocm1")
    monkeypatch.setattr(_lib, "_host", None)
    with pytest.warns(RuntimeWarning, match="built against torch"):
        assert _lib.host() is _lib.NothingOrdinary


def test_the_built_extension_is_used(monkeypatch):
    monkeypatch.setattr(_lib, "_host", None)
    assert _lib.host().__name__.endswith("._host")
