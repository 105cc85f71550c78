"""Build libmote_relation.so for gfx950 with hipcc, and the torch ops' launchers over it, in-tree.

    python -m mote_amd.build          # compile every csrc/*.hip and link mote_amd/lib/libmote_relation.so

Objects go to mote_amd/_build/, the library to mote_amd/lib/. Every call recompiles (the build
check runs it on a host without a GPU; hipcc cross-compiles). Compilation of the translation units
runs in parallel.
"""

from __future__ import annotations

import concurrent.futures as cf
import os
import shutil
import subprocess
import sys
import time

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
BUILD = os.path.join(PKG, "_build")
LIBDIR = os.path.join(PKG, "lib")
LIBNAME = "libmote_relation.so"
TORCHNAME = "_torch_launch.so"
ARCH = "gfx950"

# -packed-fp32-ops: no v_pk_{add,mul,fma}_f32 (the host pass warns that it does not know the
# feature; that is expected).
HIPFLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-fPIC",
    "-std=c++17",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I", os.path.join(ROOT, "include"),
    "-Wno-unused-result",
]


def _hipcc() -> str:
    for cand in (shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (ROCm toolchain required to build libmote_relation.so)")


def _compile(src: str) -> str:
    obj = os.path.join(BUILD, os.path.basename(src).replace(".hip", ".o"))
    cmd = [_hipcc(), *HIPFLAGS, "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {os.path.basename(src)}:\n{r.stderr[-6000:]}")
    return obj


def _build_torch_launch() -> str:
    """The torch ops' native launchers (host code over torch's headers, linked to the library beside it)."""
    import sysconfig

    import torch
    from torch.utils import cpp_extension as ce

    inc = [*ce.include_paths(), sysconfig.get_paths()["include"], os.path.join(ROOT, "include")]
    out = os.path.join(LIBDIR, TORCHNAME)
    tmp = out + ".tmp"
    cmd = [shutil.which("g++") or "g++", "-O2", "-fPIC", "-shared", "-std=c++17",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *(f"-I{p}" for p in inc),
           os.path.join(CSRC, "torch_launch.cpp"), "-o", tmp, f"-L{LIBDIR}", f"-l:{LIBNAME}",
           f"-L{os.path.join(os.path.dirname(torch.__file__), 'lib')}", "-ltorch", "-ltorch_cpu", "-ltorch_python", "-lc10",
           "-Wl,-rpath,$ORIGIN"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed on torch_launch.cpp:\n{r.stderr[-6000:]}")
    os.replace(tmp, out)
    return out


def build(verbose: bool = False) -> str:
    """Compile and link; returns the path of the shared library."""
    os.makedirs(BUILD, exist_ok=True)
    os.makedirs(LIBDIR, exist_ok=True)
    srcs = sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip"))
    t0 = time.time()
    workers = max(1, min(len(srcs), int(os.environ.get("MAX_JOBS", "8")), 16))
    with cf.ThreadPoolExecutor(workers) as ex:
        objs = list(ex.map(_compile, srcs))
    out = os.path.join(LIBDIR, LIBNAME)
    tmp = out + ".tmp"
    cmd = [_hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", *objs, "-o", tmp]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr[-4000:]}")
    os.replace(tmp, out)
    _build_torch_launch()
    if verbose:
        print(f"built {out} from {len(srcs)} sources in {time.time() - t0:.1f}s")
    return out


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
