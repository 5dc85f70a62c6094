"""Builds helmholtzbem_amd/libhbem.so (HIP for gfx950 + host setup code).

    python -m helmholtzbem_amd.build        # or: python helmholtzbem_amd/build.py

Host setup (quadrature, mass matrix, LDLT projection factor) is compiled with
g++ and -ffp-contract=off; the kernels and the C-ABI with hipcc for gfx950
(packed FP32 disabled).  Objects go to helmholtzbem_amd/_build/.
"""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libhbem.so")
ARCH = os.environ.get("HBEM_OFFLOAD_ARCH", "gfx950")

HIP_SOURCES = ["hbem_assembly.hip", "hbem_radial.hip", "hbem_dense.hip", "hbem_solve.hip", "hbem_solve_f32.hip",
               "hbem_capi.hip"]
HOST_SOURCES = ["hbem_setup.cpp"]

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
HIP_FLAGS = ["-O3", "-std=c++17", "-fPIC", "--offload-arch=" + ARCH,
             "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
             "-Wno-unused-result", "-munsafe-fp-atomics"]
HOST_FLAGS = ["-O2", "-std=c++17", "-fPIC", "-ffp-contract=off", "-march=x86-64-v2"]


def _run(cmd):
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if r.returncode != 0:
        sys.stderr.write(" ".join(cmd) + "\n" + r.stdout)
        raise RuntimeError("build step failed: " + os.path.basename(cmd[-1]))
    return r.stdout


def build(verbose: bool = False) -> str:
    os.makedirs(BUILD, exist_ok=True)
    cmds = [["g++"] + HOST_FLAGS + ["-c", os.path.join(CSRC, src), "-o", os.path.join(BUILD, src + ".o")]
            for src in HOST_SOURCES]
    cmds += [[HIPCC] + HIP_FLAGS + ["-c", os.path.join(CSRC, src), "-o", os.path.join(BUILD, src + ".o")]
             for src in HIP_SOURCES]
    with ThreadPoolExecutor(len(cmds)) as pool:
        for out in pool.map(_run, cmds):
            if verbose and out.strip():
                print(out)
    objs = [c[-1] for c in cmds]
    tmp = LIB + ".tmp"
    _run([HIPCC, "-shared", "-fPIC", "--offload-arch=" + ARCH, "-o", tmp] + objs)
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
