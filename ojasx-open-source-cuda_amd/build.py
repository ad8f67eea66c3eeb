"""Builds libojasx_e8t.so (HIP kernels + C ABI) and _ojasx_eager.so for gfx950, in-tree.

    python ojasx-open-source-cuda_amd/build.py

Objects go to ``_build/`` and the library to ``lib/libojasx_e8t.so`` next to
this file.  hipcc cross-compiles, so no GPU is needed to build.
"""

from __future__ import annotations

import concurrent.futures as cf
import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "lib", "libojasx_e8t.so")
# CPython extension of the eager calls (torch's C++ tensors over the C ABI), linked to LIB
EAGER = os.path.join(HERE, "lib", "_ojasx_eager.so")

SOURCES = [
    "e8t_codec.hip",
    "e8t_gemm_generic.hip",
    "e8t_gemm_f32.hip",
    "e8t_gemv.hip",
    "e8t_gemm_mfma.hip",
    "e8t_hadamard.hip",
    "e8t_qat.hip",
    "e8t_noalloc.hip",
    "e8t_lora.hip",
    "e8t_capi.cpp",
]

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

# Packed-fp32 VALU instructions are disabled for all device code: hipcc would
# otherwise form v_pk_*_f32 from ordinary float code.  (The host pass warns that
# it does not know the feature; that is harmless.)
DEVICE_FLAGS = ["-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
COMMON = ["-x", "hip", "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
          "-fvisibility=hidden", "-Wall", "-Wno-unused-function"] + DEVICE_FLAGS


# Per-file code generation options.  The decode GEMV keeps its MFMA results in ordinary
# VGPRs: its post-scaled kernel reads every result with VALU FMAs, and the accumulator
# register form would add a v_accvgpr_read per read and raise the register total.
EXTRA = {
    "e8t_gemv.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"],
}


def _compile(src: str) -> str:
    obj = os.path.join(BUILD, os.path.splitext(src)[0] + ".o")
    cmd = [HIPCC] + COMMON + EXTRA.get(src, []) + ["-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError(f"hipcc failed for {src}")
    return obj


def _compile_eager() -> str:
    import sysconfig

    import torch
    from torch.utils import cpp_extension

    rocm = os.path.dirname(os.path.dirname(os.path.realpath(HIPCC)))
    if not os.path.exists(os.path.join(rocm, "include", "hip", "hip_runtime.h")):
        rocm = "/opt/rocm"
    obj = os.path.join(BUILD, "e8t_torch.o")
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-w",
           "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}"]
    for d in cpp_extension.include_paths() + [os.path.join(rocm, "include"),
                                              sysconfig.get_paths()["include"]]:
        cmd += ["-isystem", d]
    r = subprocess.run(cmd + ["-c", os.path.join(CSRC, "e8t_torch.cpp"), "-o", obj],
                       capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError("g++ failed for e8t_torch.cpp")
    return obj


def _link_eager(obj: str) -> None:
    import torch

    libdir = os.path.join(os.path.dirname(torch.__file__), "lib")
    tmp = EAGER + ".tmp"
    cmd = ["g++", "-shared", "-o", tmp, obj, f"-L{libdir}", f"-L{os.path.dirname(LIB)}",
           "-l:libojasx_e8t.so", "-ltorch_python", "-ltorch", "-ltorch_cpu", "-ltorch_hip",
           "-lc10", "-lc10_hip", "-Wl,-rpath,$ORIGIN", "-Wl,--no-as-needed"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError("link of _ojasx_eager.so failed")
    os.replace(tmp, EAGER)


def build(verbose: bool = False) -> str:
    os.makedirs(BUILD, exist_ok=True)
    os.makedirs(os.path.dirname(LIB), exist_ok=True)
    with cf.ThreadPoolExecutor(max_workers=8) as ex:
        eager = ex.submit(_compile_eager)
        objs = list(ex.map(_compile, SOURCES))
        eager_obj = eager.result()
    tmp = LIB + ".tmp"
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", tmp] + objs
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError("link of libojasx_e8t.so failed")
    # a kernel template the host pass could not instantiate leaves its launch stub undefined
    # (the link of a shared library does not catch it); refuse such a library
    nm = shutil.which("nm")
    if nm:
        out = subprocess.run([nm, "-D", "--undefined-only", tmp], capture_output=True,
                             text=True).stdout
        missing = [l.split()[-1] for l in out.splitlines() if "ojx" in l]
        if missing:
            raise RuntimeError("libojasx_e8t.so has undefined symbols: " + ", ".join(missing[:4]))
    os.replace(tmp, LIB)
    _link_eager(eager_obj)
    if verbose:
        print("built", LIB)
    return LIB


if __name__ == "__main__":
    build(verbose=True)
