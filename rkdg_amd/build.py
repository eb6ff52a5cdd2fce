"""Builds the HIP library rkdg_amd/librkdg.so for gfx950 (in-tree, no JIT cache).

hipcc compiles the kernel translation units and the host C++ that implements the
C-ABI of include/rkdg_capi.h (one object per source, in parallel), then links
them; the library has no torch dependency.
"""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "librkdg.so")
SOURCES = ["rkdg_tensor.hip", "rkdg_dense.hip", "rkdg_batch.hip", "rkdg_adjoint.hip", "rkdg_noalloc.hip", "rkdg_io.hip", "rkdg_shu.hip",
           "rkdg_nc.hip", "rkdg_host.cpp", "rkdg_selftest.cpp"]
# sources built as several objects: macro and number of parts (numbered from 0)
PARTS = {"rkdg_tensor.hip": ("RKDG_TENSOR_PART", 5)}

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-result",
]


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        sys.stderr.write(res.stdout + res.stderr)
        raise RuntimeError(f"{os.path.basename(cmd[0])} failed: " + " ".join(cmd[-3:]))


def build(verbose: bool = False) -> str:
    os.makedirs(BUILD, exist_ok=True)
    objs = []
    cmds = []
    for src in SOURCES:
        macro, n = PARTS.get(src, (None, 1))
        for k in range(n):
            obj = os.path.join(BUILD, f"{src}.{k}.o" if macro else src + ".o")
            objs.append(obj)
            cmds.append([HIPCC, *FLAGS, *([f"-D{macro}={k}"] if macro else []), "-c", os.path.join(CSRC, src),
                         "-o", obj])
    with ThreadPoolExecutor(max_workers=len(cmds)) as ex:
        list(ex.map(lambda c: _run(c, verbose), cmds))
    tmp = LIB + ".tmp"
    _run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", *objs, "-o", tmp], verbose)
    os.replace(tmp, LIB)
    build_callers(verbose)
    return LIB


def build_callers(verbose: bool = False) -> None:
    """The compiled programs that the tests run: a C program on the plain header
    (gcc) and a C++ program on the class mirror include/rkdg.hpp (hipcc for the HIP
    runtime's allocation calls), which link librkdg.so, as does a third that lets HIP
    calls fail, and two that evaluate the device code's fluxes and wave speeds,
    flux_pairs with fused multiply-adds in its host half as well."""
    root = os.path.dirname(HERE)
    capi = os.path.join(root, "tests", "capi")
    if not os.path.isdir(capi):
        return
    inc = ["-I", os.path.join(root, "include"), "-I", capi]
    link = ["-L", HERE, "-lrkdg", "-Wl,-rpath,$ORIGIN/../../rkdg_amd"]
    _run(["gcc", "-std=c11", "-O2", "-Wall", *inc, os.path.join(capi, "capi_smoke.c"), *link, "-lm",
          "-o", os.path.join(capi, "capi_smoke")], verbose)
    _run([HIPCC, *FLAGS, "-Wall", *inc, os.path.join(capi, "cpp_smoke.cpp"), *link,
          "-o", os.path.join(capi, "cpp_smoke")], verbose)
    _run([HIPCC, *FLAGS, "-Wall", *inc, os.path.join(capi, "hip_faults.cpp"), *link, "-ldl",
          "-o", os.path.join(capi, "hip_faults")], verbose)
    _run([HIPCC, *FLAGS, "-Wall", "-Xarch_host", "-mfma", *inc, os.path.join(capi, "flux_pairs.hip"),
          "-o", os.path.join(capi, "flux_pairs")], verbose)
    _run([HIPCC, *FLAGS, "-Wall", *inc, os.path.join(capi, "toro_base.hip"),
          "-o", os.path.join(capi, "toro_base")], verbose)


if __name__ == "__main__":
    print(build(verbose=True))
