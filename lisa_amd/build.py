"""Builds liblisaq.so (all HIP kernels + the C ABI) and _pyops.so (the native
call path of ops.py over it) in-tree for gfx950.

Each source is compiled to an object in parallel with hipcc, then linked into
``lisa_amd/liblisaq.so``.  Compilation always runs (the driver's "does it
build" check); tests and the bench only load what is built.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
ROOT = os.path.dirname(HERE)
OUT = os.path.join(HERE, "liblisaq.so")
PYOPS = os.path.join(HERE, "_pyops.so")
OBJ = os.path.join(ROOT, "_build", "lisaq")
SOURCES = ["qmv.hip", "qmv16.hip", "qmvt.hip", "qmvd.hip", "qmvp.hip", "qmvw.hip", "qmvs.hip", "qmm.hip", "qmm_k4_p.hip", "qmm_k4_s.hip", "qmm_k2_p.hip", "qmm_k2_s.hip", "qmm_th2.hip", "qmm_th4.hip", "qmm_th8.hip", "qmm_tb8.hip", "qmm_rows_b4.hip", "qmm_rows_b28.hip", "qmm_rows_h4.hip", "qmm_rows_h28.hip", "qmm_gu.hip", "quant.hip", "qtyped.hip", "addnorm.hip", "diag.hip", "moe.hip", "moe_decode.hip", "api.cpp"]

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fvisibility=hidden",
    "-Wall",
    "-Wno-unused-function",
    # packed FP32 instructions stay off: the compiler must not form
    # v_pk_{add,mul,fma}_f32 from scalar or float2 code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I", os.path.join(ROOT, "include"),
]


def _compile(src: str) -> str:
    obj = os.path.join(OBJ, os.path.splitext(src)[0] + ".o")
    cmd = [HIPCC, *FLAGS, "-x", "hip", "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    noise = "not a recognized feature for this target"
    err = "\n".join(l for l in r.stderr.splitlines() if noise not in l and "--hip-link" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{err}")
    if err.strip():
        sys.stderr.write(err + "\n")
    return obj


def build_pyops() -> str:
    """_pyops.so: host C++ against this interpreter's torch, linked to liblisaq.so beside it."""
    import torch

    base = os.path.dirname(torch.__file__)
    inc, lib = os.path.join(base, "include"), os.path.join(base, "lib")
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1",
           "-DUSE_ROCM=1", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-isystem", inc,
           "-isystem", os.path.join(inc, "torch", "csrc", "api", "include"),
           "-I", sysconfig.get_paths()["include"], "-isystem", "/opt/rocm/include", os.path.join(CSRC, "pyops.cpp"),
           "-o", PYOPS + ".tmp", "-L" + lib, "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10", "-lc10_hip",
           "-L" + HERE, "-l:liblisaq.so", "-Wl,-rpath,$ORIGIN"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed for pyops.cpp:\n{r.stderr}")
    os.replace(PYOPS + ".tmp", PYOPS)
    return PYOPS


def build(verbose: bool = False) -> str:
    os.makedirs(OBJ, exist_ok=True)
    with cf.ThreadPoolExecutor(max_workers=min(len(SOURCES), os.cpu_count() or 4)) as ex:
        objs = list(ex.map(_compile, SOURCES))
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", OUT + ".tmp", *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    os.replace(OUT + ".tmp", OUT)
    build_pyops()
    if verbose:
        print(f"built {OUT}")
    return OUT


if __name__ == "__main__":
    build(verbose=True)
