"""Compile the HIP library in-tree for gfx950: publicrelease_2020_amd/libflosic_hip.so."""
from __future__ import annotations

import concurrent.futures
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libflosic_hip.so")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
SOURCES = ["flosic_kernels.hip", "flosic_gemm.hip", "flosic_coulomb_fp64.hip", "flosic_coulomb_fp32.hip", "flosic_coulomb_bf16.hip", "flosic_api.hip"]
HIPCC = os.path.join(ROCM, "bin", "hipcc")
OBJ = os.path.join(HERE, "_build")


def compile_command(src: str, obj: str) -> list:
    return [HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
            # packed FP32 instructions are kept out of all device code
            "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
            "-Wno-unused-command-line-argument",
            "-I" + os.path.join(ROCM, "include"), "-c", os.path.join(CSRC, src), "-o", obj]


def link_command(objs: list, out: str) -> list:
    return [HIPCC, "--offload-arch=gfx950", "-fPIC", "-shared", *objs,
            "-L" + os.path.join(ROCM, "lib"), "-lrocblas", "-Wl,-rpath," + os.path.join(ROCM, "lib"), "-o", out]


FORTRAN_EXE = os.path.join(HERE, "flosic_sic_drive")


def build_fortran(verbose: bool = False) -> str:
    """The Fortran host driver (include/flosic_hip.f90 + fortran/*.f90) linked against libflosic_hip.so."""
    fc = os.path.join(ROCM, "bin", "amdflang")
    mod = os.path.join(HERE, "_build", "fmod")
    os.makedirs(mod, exist_ok=True)
    inc = os.path.join(os.path.dirname(HERE), "include", "flosic_hip.f90")
    steps = [
        [fc, "-O2", "-J" + mod, "-c", inc, "-o", os.path.join(mod, "flosic_hip.o")],
        [fc, "-O2", "-J" + mod, "-I" + mod, "-c", os.path.join(HERE, "fortran", "flosic_sic_block.f90"), "-o",
         os.path.join(mod, "flosic_sic_block.o")],
        [fc, "-O2", "-I" + mod, os.path.join(HERE, "fortran", "flosic_sic_drive.f90"),
         os.path.join(mod, "flosic_sic_block.o"), os.path.join(mod, "flosic_hip.o"), "-L" + HERE, "-lflosic_hip",
         "-Wl,-rpath,$ORIGIN", "-o", FORTRAN_EXE + ".tmp"],
    ]
    for cmd in steps:
        if verbose:
            print(" ".join(cmd))
        res = subprocess.run(cmd, capture_output=True, text=True)
        if res.returncode != 0:
            sys.stderr.write(res.stdout + res.stderr)
            raise RuntimeError("amdflang failed building the Fortran host driver")
    os.replace(FORTRAN_EXE + ".tmp", FORTRAN_EXE)
    return FORTRAN_EXE


def _run(cmd: list, verbose: bool, what: str) -> None:
    if verbose:
        print(" ".join(cmd))
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        sys.stderr.write(res.stdout + res.stderr)
        raise RuntimeError("hipcc failed " + what)


def build(verbose: bool = False) -> str:
    """Every source in a compiler process of its own, at once; then the link."""
    os.makedirs(OBJ, exist_ok=True)
    objs = [os.path.join(OBJ, os.path.splitext(s)[0] + ".o") for s in SOURCES]
    with concurrent.futures.ThreadPoolExecutor(len(SOURCES)) as pool:
        jobs = [pool.submit(_run, compile_command(s, o), verbose, "compiling " + s) for s, o in zip(SOURCES, objs)]
        for j in jobs:
            j.result()
    tmp = LIB + ".tmp"
    _run(link_command(objs, tmp), verbose, "linking libflosic_hip.so")
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
    if os.path.exists(os.path.join(ROCM, "bin", "amdflang")):
        print(build_fortran(verbose=True))
