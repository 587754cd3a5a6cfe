"""Build recipe for libmtp_glora_amd.so (gfx950) and the torch module, in-tree.

``python -m`` is not needed: ``build_library()`` runs hipcc on every
``csrc/*.hip`` file and links them into ``lib/libmtp_glora_amd.so`` next to
this file; hipcc cross-compiles for gfx950 without a GPU present.
``build_torch_module()`` compiles ``csrc/mga_torch.cpp`` (host code only)
against the installed torch into ``lib/_mga_torch.so``.
"""
from __future__ import annotations

import hashlib
import os
import shutil
import subprocess
import sysconfig
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG_DIR = Path(__file__).resolve().parent
CSRC = PKG_DIR / "csrc"
HEADER = PKG_DIR.parent / "include" / "mtp_glora_amd.h"
LIB_DIR = PKG_DIR / "lib"
LIB_NAME = "libmtp_glora_amd.so"
TORCH_MODULE = "_mga_torch.so"
ARCH = os.environ.get("MGA_OFFLOAD_ARCH", "gfx950")

# Packed fp32 VALU ops are disabled for every device pass (hipcc's host pass
# reports the feature as unknown; that warning is harmless).
DEVICE_FLAGS = ["-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
COMMON_FLAGS = ["-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}", "-Wall",
                "-Wno-unused-function", "-Wno-unused-variable", "-munsafe-fp-atomics"]


def hipcc() -> str:
    cand = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(cand).exists():
        raise RuntimeError("hipcc not found; the ROCm toolchain is required to build libmtp_glora_amd.so")
    return cand


COMPILE_TIMEOUT_S = 900


def header_flag() -> str:
    """The C ABI's header as a number, compiled into the library and the torch module."""
    return f"-DMGA_HEADER_HASH=0x{hashlib.sha256(HEADER.read_bytes()).hexdigest()[:16]}ull"


def lib_path() -> Path:
    return LIB_DIR / LIB_NAME


def build_library(verbose: bool = False, jobs: int = 4, src_dir=None, out_path=None) -> Path:
    """Compile every csrc/*.hip to an object and link the shared library.

    src_dir / out_path build another source tree (with the same file set) into
    another library file, e.g. a variant to time against the in-tree build;
    the default is csrc/ -> lib/libmtp_glora_amd.so."""
    cc = hipcc()
    src = Path(src_dir) if src_dir is not None else CSRC
    out = Path(out_path) if out_path is not None else lib_path()
    objdir = out.parent / ("obj" if out_path is None else out.stem + "_obj")
    objdir.mkdir(parents=True, exist_ok=True)
    sources = sorted(src.glob("*.hip"))
    if not sources:
        raise RuntimeError(f"no HIP sources under {src}")

    def compile_one(src: Path) -> Path:
        obj = objdir / (src.stem + ".o")
        cmd = [cc, *COMMON_FLAGS, *DEVICE_FLAGS, header_flag(), "-c", str(src), "-o", str(obj)]
        try:
            # a compiler that loops (it has, on some unrolled kernels) fails
            # the build instead of holding it forever
            res = subprocess.run(cmd, capture_output=True, text=True, timeout=COMPILE_TIMEOUT_S)
        except subprocess.TimeoutExpired:
            raise RuntimeError(f"hipcc did not finish {src.name} within {COMPILE_TIMEOUT_S} s") from None
        if res.returncode != 0:
            raise RuntimeError(f"hipcc failed on {src.name}:\n{res.stderr}")
        if verbose:
            print(" ".join(cmd))
        return obj

    with ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(compile_one, sources))
    tmp = out.with_suffix(".so.tmp")
    # --no-undefined: a kernel template whose host launch stub the compiler
    # dropped must fail here, not when the library is loaded on a GPU box
    cmd = [cc, "-shared", f"--offload-arch={ARCH}", "-fPIC", *map(str, objs), "-o", str(tmp),
           "-L/opt/rocm/lib", "-lhipblaslt", "-Wl,--no-undefined"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr}")
    os.replace(tmp, out)
    return out


def build_torch_module(verbose: bool = False) -> Path:
    """Compile csrc/mga_torch.cpp into lib/_mga_torch.so."""
    import torch
    from torch.utils import cpp_extension
    out = LIB_DIR / TORCH_MODULE
    LIB_DIR.mkdir(parents=True, exist_ok=True)
    tmp = out.with_suffix(".so.tmp")
    include = [*cpp_extension.include_paths("cuda"), sysconfig.get_paths()["include"], "/opt/rocm/include"]
    cmd = [shutil.which("g++") or "c++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1",
           "-DUSE_ROCM=1", header_flag(), f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}",
           *(f"-isystem{p}" for p in include), str(CSRC / "mga_torch.cpp"), "-o", str(tmp),
           *(f"-L{p}" for p in cpp_extension.library_paths()), "-lc10", "-lc10_hip", "-ltorch", "-ltorch_cpu",
           "-ltorch_python"]
    res = subprocess.run(cmd, capture_output=True, text=True, timeout=COMPILE_TIMEOUT_S)
    if res.returncode != 0:
        raise RuntimeError(f"g++ failed on mga_torch.cpp:\n{res.stderr}")
    if verbose:
        print(" ".join(cmd))
    os.replace(tmp, out)
    return out


if __name__ == "__main__":
    print(build_torch_module(verbose=True))
    print(build_library(verbose=True))
