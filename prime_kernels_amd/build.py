"""Build the native library `_lib/libprime_decode.so` with hipcc for gfx950, and the host module
`_lib/_host_step-*.so` for the installed torch.

Usage: python -m prime_kernels_amd.build   (also called by __graft_entry__.build()).
The library is built in-tree so it travels with the source tree; nothing is JIT-compiled at
run time, and the Python wrappers fail loudly when it is missing.
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
LIB_DIR = PKG / "_lib"
LIB = LIB_DIR / "libprime_decode.so"
SOURCES = [PKG / "csrc" / "decode_megakernel.hip", PKG / "csrc" / "decode_sr.hip", PKG / "csrc" / "decode_cell.hip",
           PKG / "csrc" / "lossless_bf16.hip"]
HOST_SOURCE = PKG / "csrc" / "host_step.cpp"
ARCH = "gfx950"

HIPCC_FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-shared",
    # packed-fp32 ops are kept out of generated code on this target (known-unstable forms)
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-inline-asm", f"-I{ROOT / 'include'}",
    # every symbol the library uses must be defined in it
    "-Wl,--no-undefined",
]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and Path(cand).exists():
            return cand
    raise RuntimeError("hipcc not found")


def host_compiler() -> str:
    """A C++ compiler for host code: $CXX, the system's, or the clang that hipcc drives."""
    for cand in (os.environ.get("CXX"), "g++", "c++", str(Path(hipcc()).with_name("amdclang++")), "/opt/rocm/bin/amdclang++"):
        found = shutil.which(cand) if cand else None
        if found:
            return found
    raise RuntimeError("no C++ compiler found for the host module")


def build(verbose: bool = False) -> Path:
    LIB_DIR.mkdir(exist_ok=True)
    tmp = LIB.with_suffix(".so.tmp")
    cmd = [hipcc(), *HIPCC_FLAGS, *map(str, SOURCES), "-o", str(tmp)]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed ({res.returncode}):\n{res.stderr[-4000:]}")
    os.replace(tmp, LIB)
    build_host(verbose)
    return LIB


def build_host(verbose: bool = False) -> Path:
    """The Python module of the step's argument checks (host code only), against the installed torch."""
    import torch

    from prime_kernels_amd import _native

    host_lib = _native.host_path(torch.__version__)
    torch_dir = Path(torch.__file__).resolve().parent
    lib = torch_dir / "lib"
    tmp = host_lib.with_suffix(".so.tmp")
    cmd = [host_compiler(), "-O2", "-std=c++17", "-fPIC", "-shared", "-w",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", f"-I{torch_dir / 'include'}",
           f"-I{torch_dir / 'include' / 'torch' / 'csrc' / 'api' / 'include'}", f"-I{sysconfig.get_paths()['include']}",
           str(HOST_SOURCE), f"-L{lib}", "-ltorch_python", "-ltorch_cpu", "-lc10", f"-Wl,-rpath,{lib}", "-o", str(tmp)]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed ({res.returncode}):\n{res.stderr[-4000:]}")
    os.replace(tmp, host_lib)
    return host_lib


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
