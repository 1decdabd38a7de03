"""Build the wtsurf HIP library (libwtsurf.so) for gfx950 and the Fortran host, in-tree.

hipcc compiles each translation unit of csrc/ for --offload-arch=gfx950 and
links them into wannier_tools_amd/libwtsurf.so (packed-FP32 instruction
selection is switched off for all device code); amdflang then builds the
Fortran host wannier_tools_amd/bin/wt_surf against it.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libwtsurf.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"

SOURCES = ["decimate.hip", "mid.hip", "small.hip", "tiny.hip", "fourier.hip", "qpi.hip", "wtsurf_cabi.hip"]
HIPFLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # MFMA results in ordinary VGPRs: the decimation kernels budget registers
    # so that two kernels share a CU, and accumulation registers would count
    # on top of that budget
    "-mllvm", "-amdgpu-mfma-vgpr-form=1",
    "-Wall", "-Wno-unused-result",
]


def _compile(src: str) -> str:
    obj = os.path.join(BUILD, os.path.splitext(src)[0] + ".o")
    cmd = [HIPCC, *HIPFLAGS, "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stdout}\n{r.stderr}")
    return obj


FC = os.environ.get("WTSURF_FC", "/opt/rocm/llvm/bin/amdflang")
FORTRAN = os.path.join(HERE, "fortran")
BIN = os.path.join(HERE, "bin")
# order matters: modules before their users
FSOURCES = ["para_subset.f90", "wtsurf_cabi.f90", "wtsurf_dropin.f90", "wt_surf.f90"]


def build_fortran(verbose: bool = False) -> str:
    """The Fortran host: wt_surf linked against libwtsurf.so (rpath to it)."""
    mod = os.path.join(BUILD, "fmod")
    os.makedirs(mod, exist_ok=True)
    os.makedirs(BIN, exist_ok=True)
    objs = []
    for src in FSOURCES:
        obj = os.path.join(mod, os.path.splitext(src)[0] + ".o")
        cmd = [FC, "-O2", "-fPIC", "-module-dir", mod, "-c", os.path.join(FORTRAN, src), "-o", obj]
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"amdflang failed for {src}:\n{r.stdout}\n{r.stderr}")
        objs.append(obj)
    exe = os.path.join(BIN, "wt_surf")
    cmd = [FC, "-o", exe, *objs, f"-L{HERE}", "-lwtsurf", "-Wl,-rpath,$ORIGIN/.."]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link of wt_surf failed:\n{r.stdout}\n{r.stderr}")
    if verbose:
        print(f"built {exe}")
    return exe


def build(verbose: bool = False) -> str:
    os.makedirs(BUILD, exist_ok=True)
    with cf.ThreadPoolExecutor(max_workers=len(SOURCES)) as ex:
        objs = list(ex.map(_compile, SOURCES))
    tmp = LIB + ".tmp"
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB)
    if verbose:
        print(f"built {LIB}")
    build_fortran(verbose)
    return LIB


if __name__ == "__main__":
    build(verbose="-q" not in sys.argv)
