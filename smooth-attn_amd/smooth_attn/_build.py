"""Build recipe for the HIP library ``libsmooth_attn_amd.so`` (gfx950 only) and
the Python extension ``_host`` (the native call path, host code only).

Each ``csrc/*.hip`` file is compiled by ``hipcc --offload-arch=gfx950`` in
parallel and linked into one shared library placed next to this file, so it
travels with the source tree; ``csrc/host/host.cpp`` is compiled against the
installed torch beside it.  Run ``python -m smooth_attn._build`` (with
``smooth-attn_amd`` on ``sys.path``) or call :func:`build`.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import shutil
import subprocess
import sys
from pathlib import Path

PKG_DIR = Path(__file__).resolve().parent
CSRC = PKG_DIR.parent / "csrc"
INCLUDE = PKG_DIR.parent.parent / "include"
LIB_NAME = "libsmooth_attn_amd.so"
HOST_NAME = "_host.so"
OBJ_DIR = PKG_DIR.parent / "_build"

ARCH = "gfx950"
HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-ffp-contract=fast",
    "-munsafe-fp-atomics",
    # Packed FP32 (v_pk_*_f32) is kept out of all generated code.
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def _hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and Path(cand).exists():
            return cand
    raise RuntimeError("hipcc not found: the smooth_attn HIP library cannot be built")


def _compile(src: Path, hipcc: str, verbose: bool) -> Path:
    obj = OBJ_DIR / (src.stem + ".o")
    cmd = [hipcc, *HIPCC_FLAGS, f"-I{INCLUDE}", f"-I{CSRC}", "-c", str(src), "-o", str(obj)]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src.name}:\n{res.stderr}")
    return obj


def _build_host(hipcc: str, verbose: bool) -> Path:
    """Compile csrc/host/host.cpp against torch into the extension ``_host.so``."""
    import sysconfig

    from torch.utils import cpp_extension

    out = PKG_DIR / HOST_NAME
    tmp = out.with_suffix(".so.tmp")
    rocm = Path(hipcc).resolve().parent.parent
    libs = cpp_extension.library_paths()
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1",
           "-DUSE_ROCM", f"-D_GLIBCXX_USE_CXX11_ABI={int(_torch_cxx11_abi())}", f"-I{INCLUDE}",
           *(f"-isystem{p}" for p in cpp_extension.include_paths()), f"-isystem{rocm / 'include'}",
           "-isystem/opt/rocm/include", f"-isystem{sysconfig.get_paths()['include']}",
           str(CSRC / "host" / "host.cpp"), "-o", str(tmp),
           *(f"-L{p}" for p in libs), "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python"]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"g++ failed for host.cpp:\n{res.stderr}")
    os.replace(tmp, out)
    return out


def _torch_cxx11_abi() -> bool:
    import torch

    return torch.compiled_with_cxx11_abi()


def build(verbose: bool = False, jobs: int | None = None) -> Path:
    """Compile every csrc/*.hip for gfx950 and link the shared library, and
    compile the host extension."""
    hipcc = _hipcc()
    OBJ_DIR.mkdir(exist_ok=True)
    sources = sorted(CSRC.glob("*.hip"))
    if not sources:
        raise RuntimeError(f"no HIP sources under {CSRC}")
    jobs = jobs or min(8, len(sources))
    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        host = ex.submit(_build_host, hipcc, verbose)
        objs = list(ex.map(lambda s: _compile(s, hipcc, verbose), sources))
        host.result()
    out = PKG_DIR / LIB_NAME
    tmp = out.with_suffix(".so.tmp")
    cmd = [hipcc, f"--offload-arch={ARCH}", "-shared", "-fPIC", *map(str, objs), "-o", str(tmp)]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr}")
    os.replace(tmp, out)
    return out


if __name__ == "__main__":
    path = build(verbose="-v" in sys.argv)
    print(path)
