"""Build libtq_hip.so (the gfx950 kernels + C ABI) and _tq_torch.so (torch's
side of it: the ops' C++ kernels) in-tree with hipcc.

    python -m turboquant_amd.build

Both land next to this file so they travel with the source tree; the loaders
(turboquant_amd._lib, turboquant_amd.ops) never build implicitly on a GPU host.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libtq_hip.so")
TORCH_LIB = os.path.join(HERE, "_tq_torch.so")
SOURCES = ["tq_write.hip", "tq_decode.hip", "tq_dequant.hip", "tq_prefill.hip", "tq_mse.hip",
           "tq_qjl.hip", "tq_e2e.hip"]
ARCH = os.environ.get("TQ_OFFLOAD_ARCH", "gfx950")

HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-shared",
    # packed fp32 VALU forms are kept out of every kernel
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # IEEE division and sqrt (the write kernel's bit parity relies on them)
    "-fno-fast-math",
    "-fhip-fp32-correctly-rounded-divide-sqrt",
    "-Wall",
    "-Wno-unused-function",
]


def hipcc() -> str:
    for c in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if c and os.path.exists(c):
            return c
    raise RuntimeError("hipcc not found")


def _run(cmd, tmp: str, out: str, verbose: bool) -> str:
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed ({r.returncode}):\n{r.stdout}\n{r.stderr}")
    if verbose and r.stderr.strip():
        print(r.stderr, file=sys.stderr)
    os.replace(tmp, out)
    return out


def build_torch(verbose: bool = False) -> str:
    """_tq_torch.so: host code only, against the installed torch's headers and
    libraries and libtq_hip.so beside it (built first)."""
    import sysconfig

    import torch
    from torch.utils.cpp_extension import include_paths, library_paths
    tmp = TORCH_LIB + ".tmp"
    libs = [p for d in library_paths() for p in (f"-L{d}", f"-Wl,-rpath,{d}")]
    cmd = [hipcc(), "-x", "c++", "-O2", "-std=c++17", "-fPIC", "-shared",
           "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           *[f"-isystem{d}" for d in (*include_paths(), sysconfig.get_paths()["include"],
                                      "/opt/rocm/include")],
           os.path.join(CSRC, "tq_torch.cpp"), "-x", "none", LIB, "-Wl,-rpath,$ORIGIN", *libs,
           "-lc10", "-ltorch", "-ltorch_cpu", "-ltorch_python", "-lc10_hip", "-o", tmp]
    return _run(cmd, tmp, TORCH_LIB, verbose)


def build(verbose: bool = False) -> str:
    srcs = [os.path.join(CSRC, s) for s in SOURCES]
    tmp = LIB + ".tmp"
    cmd = [hipcc(), *HIPCC_FLAGS, *srcs, "-Wl,-soname,libtq_hip.so", "-o", tmp]
    _run(cmd, tmp, LIB, verbose)
    build_torch(verbose)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
