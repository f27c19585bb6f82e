"""Build libbytes_amd.so (all HIP kernels + the C ABI) in-tree for gfx950, and
_native.so, the operators' native call path over it.

    python -m bytes_amd.build            # compile every csrc/*.hip, link the .so files

The libraries are placed next to this file so that they travel with the source
tree; nothing is installed anywhere else.
"""
from __future__ import annotations

import concurrent.futures as cf
import glob
import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libbytes_amd.so")
NATIVE = os.path.join(HERE, "_native.so")       # the operators' native call path (host code)
ARCH = "gfx950"

HIPCC = os.environ.get("HIPCC") or shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

CFLAGS = [
    "-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}",
    # Packed FP32 VALU forms are kept out of every kernel.
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unused-variable",
    "-I", CSRC,
]


def _compile(src: str) -> str:
    obj = os.path.join(OBJ, os.path.basename(src) + ".o")
    cmd = [HIPCC, *CFLAGS, "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stdout}\n{r.stderr}")
    return obj


def _link(objs: list) -> str:
    """libbytes_amd.so from the kernels' objects, in the build folder."""
    out = os.path.join(OBJ, os.path.basename(LIB))
    r = subprocess.run([HIPCC, "-shared", "-fPIC", f"--offload-arch={ARCH}", "-o", out, *objs], capture_output=True,
                       text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    return out


def _compile_native() -> str:
    """The extension module csrc/host/native.cpp, in the build folder: host code
    against torch's headers, linked to the libbytes_amd.so beside it."""
    import sysconfig

    import torch
    from torch.utils import cpp_extension as C
    cxx = os.environ.get("CXX") or shutil.which("g++") or "/opt/rocm/llvm/bin/clang++"
    out = os.path.join(OBJ, os.path.basename(NATIVE))
    cmd = [cxx, "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           *(f"-isystem{p}" for p in C.include_paths()), "-isystem/opt/rocm/include",
           f"-isystem{sysconfig.get_paths()['include']}", os.path.join(CSRC, "host", "native.cpp"), "-o", out,
           *(f"-L{p}" for p in C.library_paths()), "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10", "-lc10_hip",
           f"-L{OBJ}", f"-l:{os.path.basename(LIB)}", "-Wl,-rpath,$ORIGIN"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"{cxx} failed for csrc/host/native.cpp:\n{r.stdout}\n{r.stderr}")
    return out


def build(verbose: bool = False) -> str:
    os.makedirs(OBJ, exist_ok=True)
    srcs = sorted(glob.glob(os.path.join(CSRC, "*.hip")))
    if not srcs:
        raise RuntimeError("no HIP sources found")
    workers = max(1, min(len(srcs), int(os.environ.get("MAX_JOBS", os.cpu_count() or 4))))
    with cf.ThreadPoolExecutor(workers) as ex:
        objs = list(ex.map(_compile, srcs))
    lib = _link(objs)
    native = _compile_native()
    # both are built: the pair beside this file is replaced as one.  The old
    # extension goes first, so that none is ever beside a library of another
    # version, whose entry points may take other arguments.
    if os.path.exists(NATIVE):
        os.remove(NATIVE)
    os.replace(lib, LIB)
    os.replace(native, NATIVE)
    if verbose:
        print(f"built {LIB} from {len(srcs)} sources and {NATIVE}")
    return LIB


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
