"""Builds libmortar_hip.so (gfx950 kernels and the C-ABI) and _mortar_native.so (the call layer between torch and it) in-tree
with hipcc.  `python build.py` or mortar_amd.build.build()."""
from __future__ import annotations

import os
import shutil
import subprocess
import sys

_HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(_HERE, "csrc")
LIB = os.path.join(_HERE, "libmortar_hip.so")
NATIVE = os.path.join(_HERE, "_mortar_native.so")
SOURCES = ["mortar_host.cpp", "mortar_prefill.hip", "mortar_smallm.hip", "mortar_smallm_chunk.hip", "mortar_mid.hip", "mortar_pipe.hip", "mortar_decode.hip", "mortar_gemv_f32.hip", "mortar_route.hip", "mortar_router_gemm.hip",
           "mortar_pack.hip", "mortar_sdd.hip", "mortar_swiglu.hip", "mortar_values.hip"]
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]


def _native_flags(hipcc: str) -> tuple:
    """(compile, link) flags of the host-only call layer: torch's headers and libraries."""
    import sysconfig

    import torch
    from torch.utils.cpp_extension import include_paths
    libs = os.path.join(os.path.dirname(torch.__file__), "lib")
    return (["-O2", "-std=c++17", "-fPIC", "-w", "-x", "c++", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
             f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
             *(f"-I{d}" for d in (*include_paths(), sysconfig.get_paths()["include"])),
             "-I" + os.path.join(os.path.dirname(os.path.dirname(os.path.realpath(hipcc))), "include")],
            [f"-L{libs}", "-ltorch", "-ltorch_cpu", "-ltorch_python", "-lc10", "-lc10_hip", "-Wl,-rpath,$ORIGIN"])


def build(verbose: bool = False) -> str:
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        raise RuntimeError("hipcc not found: cannot build libmortar_hip.so")
    objs = []
    procs = []
    for src in SOURCES:
        obj = os.path.join(CSRC, os.path.splitext(src)[0] + ".o")
        cmd = [hipcc, *FLAGS, "-x", "hip", "-c", os.path.join(CSRC, src), "-o", obj]
        procs.append((src, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)))
        objs.append(obj)
    nflags, nlink = _native_flags(hipcc)
    nobj = os.path.join(CSRC, "mortar_torch.o")
    procs.append(("mortar_torch.cpp", subprocess.Popen([hipcc, *nflags, "-c", os.path.join(CSRC, "mortar_torch.cpp"), "-o", nobj],
                                                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)))
    for src, pr in procs:
        out, _ = pr.communicate()
        if pr.returncode != 0:
            raise RuntimeError(f"hipcc failed on {src}:\n{out}")
        if verbose and out.strip():
            print(out)
    subprocess.check_call([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-Wl,-soname,libmortar_hip.so", "-o", LIB, *objs])
    subprocess.check_call([hipcc, "-shared", "-fPIC", "-o", NATIVE, nobj, LIB, *nlink])
    return LIB


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
