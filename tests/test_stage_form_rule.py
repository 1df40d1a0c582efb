"""Which parts an FP64 stage launch runs (16x4x2 or 16x4x4), by its form and its size: fixed forms hold
only where every block's rows and buffers allow them, as a level reports it; others go by the launch's
size. Host-only: the rule is called in the built library."""
import ctypes as C
import os
import subprocess

import pytest

import granite_amd as ga
from granite_amd import ccz4

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = """
#include "kernels.hpp"
extern "C" int large(int variant, int pairs_ok, int ntiles) {
    gr::Batch B{};
    B.variant = variant;
    B.pairs_ok = pairs_ok;
    B.ntiles = ntiles;
    return gr::stage_parts_large(B);
}
"""


@pytest.fixture(scope="module")
def large(tmp_path_factory):
    try:
        ga.library()
    except Exception as exc:
        pytest.skip(f"library not available: {exc}")
    d = tmp_path_factory.mktemp("form")
    (d / "form.cpp").write_text(SRC)
    lib = ccz4.library_path()
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I",
                    os.path.join(ROOT, "granite_amd", "csrc"), str(d / "form.cpp"), lib,
                    "-Wl,-rpath," + os.path.dirname(lib), "-o", str(d / "form.so")], check=True)
    return C.CDLL(str(d / "form.so")).large


@pytest.mark.parametrize("ntiles,by_size", [(1, 0), (64, 0), (65, 1), (4096, 1)])
def test_rule(large, ntiles, by_size):
    for pairs_ok in (0, 1):
        assert large(0, pairs_ok, ntiles) == by_size
    assert (large(1, 1, ntiles), large(2, 1, ntiles)) == (0, 1)
    assert (large(1, 0, ntiles), large(2, 0, ntiles)) == (by_size, by_size)
