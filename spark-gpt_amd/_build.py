"""Build recipe for ``libsparkfp8.so`` (hand-written gfx950 HIP kernels behind
a C ABI, compiled in-tree with hipcc) and ``_native.so`` (the torch-facing
wrappers of a step's calls, host code compiled with g++ against torch's
headers and linked to the former); no torch extension machinery.

Usage: ``python spark-gpt_amd/_build.py`` or ``build()`` from Python.
"""
from __future__ import annotations

import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libsparkfp8.so")
SOURCES = ("quant.hip", "gemm.hip", "moe.hip", "bf16.hip", "optim.hip")
NATIVE = os.path.join(HERE, "_native.so")
NATIVE_SOURCE = "native.cpp"
ARCH = "gfx950"

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    # packed fp32 ops are disabled for every kernel of this library
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


CXX = os.environ.get("CXX", "g++")


def _native_compile() -> list[str]:
    import sysconfig

    import torch

    inc = os.path.join(os.path.dirname(torch.__file__), "include")
    rocm = os.path.join(os.path.dirname(os.path.dirname(HIPCC)), "include")
    return [CXX, "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-w",
            f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-D__HIP_PLATFORM_AMD__=1",
            "-DUSE_ROCM=1", f"-I{inc}", f"-I{os.path.join(inc, 'torch', 'csrc', 'api', 'include')}", f"-I{rocm}",
            f"-I{sysconfig.get_paths()['include']}"]


def _native_link() -> list[str]:
    import torch

    lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    return [f"-L{lib}", "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python", f"-L{HERE}", "-lsparkfp8",
            "-Wl,-rpath,$ORIGIN"]


def _run(cmd: list[str]) -> None:
    proc = subprocess.run(cmd, cwd=CSRC, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"build failed: {' '.join(cmd)}\n{proc.stdout}\n{proc.stderr}")


def build(verbose: bool = False) -> str:
    """Compile every source for gfx950, link ``libsparkfp8.so`` and then
    ``_native.so`` against it; returns the path of the former."""
    from concurrent.futures import ThreadPoolExecutor

    objs = [os.path.join(CSRC, os.path.splitext(s)[0] + ".o") for s in SOURCES]
    cmds = [[HIPCC, *FLAGS, "-c", src, "-o", obj] for src, obj in zip(SOURCES, objs)]
    native_obj = os.path.join(CSRC, "native.o")
    cmds.append([*_native_compile(), "-c", NATIVE_SOURCE, "-o", native_obj])
    with ThreadPoolExecutor(max_workers=len(cmds)) as ex:
        list(ex.map(_run, cmds))
    tmp = LIB + ".tmp"
    _run([HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs])
    os.replace(tmp, LIB)
    tmp = NATIVE + ".tmp"
    _run([CXX, "-shared", "-o", tmp, native_obj, *_native_link()])
    os.replace(tmp, NATIVE)
    for o in [*objs, native_obj]:
        os.remove(o)
    if verbose:
        print(f"built {LIB} and {NATIVE}", file=sys.stderr)
    return LIB


if __name__ == "__main__":
    build(verbose=True)
