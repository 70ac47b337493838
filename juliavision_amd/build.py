"""Builds ``libmi355dnn.so`` (the C-ABI library of HIP kernels) in-tree for gfx950.

``hipcc`` cross-compiles without a GPU, so this runs on a CPU-only build host;
the resulting shared object sits next to this file.  ``_host.so`` beside it is the native host side of ``kernels.py``
(csrc/host.cpp: plain C++ over torch's headers, linked against the library).
"""
from __future__ import annotations

import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libmi355dnn.so")
HOST = os.path.join(HERE, "_host.so")
SOURCES = ["gemm.hip", "gemm_skinny.hip", "gemm_pipe.hip", "gemm_ring.hip", "gemm_deep.hip", "gemm_any.hip", "sdpa.hip", "sdpa_tile.hip", "sdpa_decode.hip", "conv.hip", "conv_tile.hip", "convtranspose.hip", "layernorm.hip", "kvcache.hip", "layout.hip", "probe.hip"]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
# -packed-fp32-ops: keep the compiler from forming v_pk_*_f32 out of scalar float code.
# -Xarch_device -fno-honor-nans: no kernel relies on NaN propagation (infinities stay honoured: they are the masks);
#   without it every fmaxf operand is first canonicalised with an extra v_max_f32.  Device code only: the host side
#   checks its arguments with ordinary IEEE comparisons.
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-Xarch_device", "-fno-honor-nans",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-Wno-unused-command-line-argument"]


def _compile(src: str) -> str:
    obj = os.path.join(CSRC, src.replace(".hip", ".o"))
    cmd = [HIPCC, *FLAGS, "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in r.stderr.splitlines() if "is not a recognized feature" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{err}")
    if err.strip():
        sys.stderr.write(err + "\n")
    return obj


def _compile_host() -> str:
    from torch.utils.cpp_extension import include_paths
    import torch
    obj = os.path.join(CSRC, "host.o")
    inc = [f"-I{p}" for p in include_paths() + [sysconfig.get_paths()["include"], "/opt/rocm/include"]]
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           "-Wno-attributes", *inc, "-c", os.path.join(CSRC, "host.cpp"), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed on host.cpp:\n{r.stderr}")
    return obj


def _link_host(obj: str) -> None:
    from torch.utils.cpp_extension import library_paths
    cmd = ["g++", "-shared", "-o", HOST, obj, f"-L{HERE}", "-Wl,-rpath,$ORIGIN", "-l:libmi355dnn.so", *[f"-L{p}" for p in library_paths()],
           "-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link of _host.so failed:\n{r.stderr}")


def build(verbose: bool = True) -> str:
    with ThreadPoolExecutor(max_workers=8) as ex:
        host = ex.submit(_compile_host)
        objs = list(ex.map(_compile, SOURCES))
        host_obj = host.result()
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    _link_host(host_obj)
    if verbose:
        print(f"built {LIB} and {HOST}")
    return LIB


if __name__ == "__main__":
    build()
