"""Builds libm2_amd.so (gfx950) from m2_amd/csrc with hipcc, in-tree.

    python m2_amd/build.py                 # compile every .hip and link
    python m2_amd/build.py --incremental   # recompile only the sources that changed
"""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libm2_amd.so")
SOURCES = ["common.hip", "fftconv_kernels.hip", "fftconv_real_kernels.hip", "fftconv_long_kernels.hip", "mixer_taps_kernels.hip", "hyena_filter_kernels.hip", "filter_fused_kernels.hip", "blockdiag_kernels.hip", "wo_layernorm_kernels.hip",
           "mlp_fused_kernels.hip", "glu_stream_kernels.hip", "dense_kernels.hip", "dense_ws_kernels.hip", "split_gemm_kernels.hip", "layernorm_kernels.hip", "pooler_kernels.hip", "encoder_schedule.hip"]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
# packed fp32 VALU instructions are switched off on purpose (device flag, the host pass warns about it)
FLAGS = ["-std=c++17", "-O3", "--offload-arch=gfx950", "-fPIC", "-Xclang", "-target-feature", "-Xclang",
         "-packed-fp32-ops", "-Wno-unused-command-line-argument"]


def _up_to_date(obj: str) -> bool:
    if not os.path.exists(obj):
        return False
    t = os.path.getmtime(obj)
    deps = [os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".h")]
    deps += [os.path.join(CSRC, os.path.splitext(os.path.basename(obj))[0] + ".hip"),
             os.path.join(HERE, "..", "include", "m2_amd.h"), os.path.abspath(__file__)]
    return all(os.path.getmtime(d) < t for d in deps)


def _compile(src: str, incremental: bool = False) -> str:
    obj = os.path.join(CSRC, os.path.splitext(src)[0] + ".o")
    if incremental and _up_to_date(obj):
        return obj
    cmd = [HIPCC, *FLAGS, "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{err}")
    if err.strip():
        sys.stderr.write(err + "\n")
    return obj


def _build_param_check(incremental: bool = False) -> str:
    """m2_amd/_param_check.so, a host-only CPython extension against torch's headers."""
    import sysconfig

    import torch
    from torch.utils.cpp_extension import include_paths, library_paths
    src, out = os.path.join(CSRC, "param_check.cpp"), os.path.join(HERE, "_param_check.so")
    if incremental and os.path.exists(out) and os.path.getmtime(src) < os.path.getmtime(out):
        return out
    cmd = ["g++", "-std=c++17", "-O2", "-fPIC", "-shared", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           *[f"-I{p}" for p in include_paths()], f"-I{sysconfig.get_paths()['include']}", src, "-o", out,
           *[f"-L{p}" for p in library_paths()], "-lc10", "-ltorch_cpu", "-ltorch_python"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed for param_check.cpp:\n{r.stderr}")
    return out


def build(verbose: bool = True, incremental: bool = False) -> str:
    """Compiles every source (or, with incremental=True, only those older than their .hip / headers) and links."""
    with ThreadPoolExecutor(max_workers=min(8, len(SOURCES))) as ex:
        check = ex.submit(_build_param_check, incremental)
        objs = list(ex.map(lambda src: _compile(src, incremental), SOURCES))
        check.result()
    cmd = [HIPCC, "-shared", "-fPIC", "--offload-arch=gfx950", "-o", LIB, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    if verbose:
        print(f"built {LIB}")
    return LIB


if __name__ == "__main__":
    build(incremental="--incremental" in sys.argv)
