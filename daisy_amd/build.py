"""Builds ``libdaisy_hip.so`` (the gfx950 kernels + C ABI) in-tree with hipcc.

Run as ``python -m daisy_amd.build``.  hipcc cross-compiles for gfx950 without
a GPU, so this works on a CPU-only machine; the resulting library sits next to
the sources so that it travels with the tree.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "csrc")
LIB_NAME = "libdaisy_hip.so"
LIB_PATH = os.path.join(CSRC, LIB_NAME)
SOURCES = ["abi.hip", "decode.hip", "prefill.hip", "kda.hip", "kda_step.hip", "prep.hip", "proj.hip", "kimi.hip", "linear.hip", "layer_step.hip"]
# Diagnostic kernels of the benchmark (matrix-pipe and read-stream ceilings): not part of the product.  Their source
# sits next to bench.py at the repository root and is built into a library of its own there, which only bench.py loads.
ROOT = os.path.dirname(os.path.dirname(CSRC))
PROBE_LIB_NAME = "libdaisy_bench_probe.so"
PROBE_LIB_PATH = os.path.join(ROOT, PROBE_LIB_NAME)
PROBE_SOURCE = os.path.join(ROOT, "bench_probe.hip")

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fno-gpu-rdc",
    "-Wall",
    "-Wno-unused-function",
    # Keep the compiler from forming packed-fp32 instructions from scalar code.
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found (looked on PATH and in /opt/rocm/bin)")
    return exe


def _compile(src: str, verbose: bool) -> str:
    path = src if os.path.isabs(src) else os.path.join(CSRC, src)
    obj = os.path.splitext(path)[0] + ".o"
    cmd = [_hipcc(), *HIPCC_FLAGS, "-I", ROOT, "-c", path, "-o", obj]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{r.stdout}\n{r.stderr}")
    if verbose and r.stderr.strip():
        # The host pass warns that it does not know the packed-fp32 feature; harmless.
        lines = [ln for ln in r.stderr.splitlines() if "packed-fp32-ops" not in ln]
        if lines:
            print("\n".join(lines), flush=True)
    return obj


# The call path from torch tensors to the kernels (a CPython extension linked against the product library and torch).
NATIVE_SOURCE = os.path.join(CSRC, "native.cpp")
NATIVE_PATH = os.path.join(os.path.dirname(CSRC), "_native.so")


def _native_command() -> list:
    """The host compiler with the flags of native.cpp: every warning on for our code, headers of others (-isystem) quiet."""
    import sysconfig
    import torch
    from torch.utils.cpp_extension import include_paths
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-Wall", "-Wextra", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}"]
    for inc in (*include_paths(), "/opt/rocm/include", sysconfig.get_paths()["include"]):
        cmd += ["-isystem", inc]
    return cmd


def _compile_native(verbose: bool) -> str:
    obj = os.path.splitext(NATIVE_SOURCE)[0] + ".o"
    _run([*_native_command(), "-c", NATIVE_SOURCE, "-o", obj], "native.cpp", verbose)
    return obj


def _link_native(obj: str, verbose: bool) -> None:
    import torch
    lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    _run(["g++", "-shared", "-o", NATIVE_PATH, obj, "-L", CSRC, f"-l:{LIB_NAME}", "-Wl,-rpath,$ORIGIN/csrc", "-L", lib,
          "-ltorch_python", "-ltorch_hip", "-ltorch_cpu", "-ltorch", "-lc10_hip", "-lc10"], "native.cpp", verbose)


def _run(cmd, what: str, verbose: bool) -> None:
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"building {what} failed:\n{r.stdout}\n{r.stderr}")
    if verbose and r.stderr.strip():
        print(r.stderr, flush=True)


def _link(objs, out: str, verbose: bool) -> None:
    cmd = [_hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-fno-gpu-rdc", *objs, "-o", out]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")


def build(verbose: bool = True, sources=None) -> str:
    """Compiles every source and links the product library (and the benchmark's probe library);
    returns the product library's path."""
    srcs = list(sources or SOURCES)
    every = srcs + ([PROBE_SOURCE] if os.path.exists(PROBE_SOURCE) else [])
    if "abi.hip" not in every:
        every.append("abi.hip")
    with ThreadPoolExecutor(max_workers=min(6, len(every) + 1)) as ex:
        native = ex.submit(_compile_native, verbose)
        objs = dict(zip(every, ex.map(lambda s: _compile(s, verbose), every)))
    _link([objs[s] for s in srcs], LIB_PATH, verbose)
    _link_native(native.result(), verbose)
    if PROBE_SOURCE in objs:
        _link([objs["abi.hip"], objs[PROBE_SOURCE]], PROBE_LIB_PATH, verbose)
    return LIB_PATH


if __name__ == "__main__":
    print(build(verbose="-q" not in sys.argv))
