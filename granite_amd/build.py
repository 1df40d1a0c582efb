"""Build recipe of the HIP engine: gfx950 code objects + C ABI in one shared library.

    python -m granite_amd.build        (or granite_amd.build.build())

The library is written in-tree as granite_amd/libgranite_ccz4.so.
"""
from __future__ import annotations

import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
LIB = os.path.join(HERE, "libgranite_ccz4.so")
SOURCES = [os.path.join(HERE, "csrc", f) for f in ("kernels.hip", "capi.hip")]
HEADERS = [os.path.join(HERE, "csrc", f) for f in ("kernels.hpp", "ccz4_cell.hpp")] + [
    os.path.join(ROOT, "include", "granite_ccz4.h")
]

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-shared",
    # packed-FP32 instructions stay disabled for all device code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
    "-Wl,-soname,libgranite_ccz4.so",
]


def build(verbose: bool = False, out: str = LIB, defines=()) -> str:
    """Compile every source into `out` (default: the in-tree library); always recompiles.
    `defines` are extra -D macros (tile shape of the stage kernels)."""
    tmp = out + ".tmp"
    cmd = [HIPCC, *FLAGS, *["-D" + d for d in defines], "-I", os.path.join(ROOT, "include"), *SOURCES, "-o", tmp]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("hipcc failed:\n" + res.stdout + res.stderr)
    os.replace(tmp, out)
    return out


DRIVER_SRC = os.path.join(HERE, "host", "granite_main.cpp")
DRIVER = os.path.join(HERE, "bin", "granite_main")
# where the reference's launcher looks for the binary (scripts/run_granite.py:292-297, with its
# default build directory "build"), so that launcher runs this driver unchanged from the repo root
DRIVER_LAUNCHER = os.path.join(ROOT, "build", "bin", "granite_main")


def build_driver(verbose: bool = False, lib: str = LIB, out: str = DRIVER) -> str:
    """The granite_main driver (host C++17 over the C ABI), linked to the in-tree library
    (found at run time through $ORIGIN, so the tree can move). Built at `out` and, for the
    default output, also at build/bin/granite_main."""
    if out == DRIVER:
        _link_driver(verbose, lib, DRIVER_LAUNCHER)
    return _link_driver(verbose, lib, out)


def _link_driver(verbose: bool, lib: str, out: str) -> str:
    os.makedirs(os.path.dirname(out), exist_ok=True)
    cxx = os.environ.get("CXX", "g++")
    tmp = out + ".tmp"
    cmd = [cxx, "-std=c++17", "-O2", "-Wall", "-I", os.path.join(ROOT, "include"), "-I", os.path.join(HERE, "host"),
           DRIVER_SRC, "-L", os.path.dirname(lib), "-lgranite_ccz4",
           "-Wl,-rpath,$ORIGIN/" + os.path.relpath(os.path.dirname(lib), os.path.dirname(out)),
           "-Wl,-rpath-link,/opt/rocm/lib", "-o", tmp]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("driver build failed:\n" + res.stdout + res.stderr)
    os.replace(tmp, out)
    return out


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
    print(build_driver(verbose="-v" in sys.argv))
