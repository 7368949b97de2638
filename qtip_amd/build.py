"""Compile libqtip_hip.so for gfx950 and the host module in-tree:  python -m qtip_amd.build"""
import os
import subprocess
import sys
import tempfile
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
SRCS = [os.path.join(HERE, "csrc", f)
        for f in ("qtip_hip.hip", "qtip_gemm.hip", "qtip_rht.hip", "qtip_decoder.hip", "qtip_pack.hip", "qtip_prefill.hip", "qtip_train.hip",
                  "qtip_linear.hip", "qtip_head.hip")]
OUT = os.path.join(HERE, "libqtip_hip.so")
HOST_SRC = os.path.join(HERE, "csrc", "qtip_host.cpp")
HOST_OUT = os.path.join(HERE, "_qtip_host.so")

# packed fp32 VALU forms are switched off for every HIP translation unit
HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in res.stderr.splitlines() if "packed-fp32-ops" not in l)
    if res.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed:\n{err}")
    if err.strip() and verbose:
        print(err, file=sys.stderr)


def compile_library(out, extra=(), verbose=True):
    """The library's sources, compiled side by side (hipcc takes them one after the other), into `out`."""
    hipcc = os.environ.get("HIPCC", "hipcc")
    with tempfile.TemporaryDirectory() as tmp, ThreadPoolExecutor(len(SRCS)) as pool:
        objs = [os.path.join(tmp, os.path.basename(s) + ".o") for s in SRCS]
        list(pool.map(lambda so: _run([hipcc] + HIPCC_FLAGS + list(extra) + ["-c", so[0], "-o", so[1]], verbose),
                      zip(SRCS, objs)))
        _run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC"] + objs + ["-o", out + ".tmp"], verbose)
    os.replace(out + ".tmp", out)
    return out


def build_host(verbose=True):
    """The native side of the wrappers' short ways (no device code), against the installed torch."""
    import sysconfig

    import torch
    from torch.utils.cpp_extension import include_paths
    dirs = include_paths() + [sysconfig.get_paths()["include"]]
    _run([os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared",
          f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", f'-DQTIP_TORCH_VERSION="{torch.__version__}"'] + [a for d in dirs for a in ("-isystem", d)] +
         [HOST_SRC, "-L" + os.path.join(os.path.dirname(torch.__file__), "lib"), "-ltorch_python", "-ltorch_cpu", "-lc10",
          "-o", HOST_OUT + ".tmp"], verbose)
    os.replace(HOST_OUT + ".tmp", HOST_OUT)
    return HOST_OUT


def build(verbose=True):
    build_host(verbose)
    return compile_library(OUT, verbose=verbose)


if __name__ == "__main__":
    build()
