"""Host arithmetic of the screened searches (px_host.h), compiled as it is into a small library
and checked on the CPU."""
import ctypes
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "proxima_amd", "csrc")

SHIM = r"""
#include "px_host.h"
extern "C" {
int64_t ref_roundings(int64_t n) { return px::ref_roundings(n); }
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("screen_host")
    src, out = d / "shim.cpp", d / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-I", CSRC, "-o", str(out),
                    str(src), "-lpthread"], check=True, timeout=120)
    lib = ctypes.CDLL(str(out))
    lib.ref_roundings.restype = ctypes.c_int64
    lib.ref_roundings.argtypes = [ctypes.c_int64]
    return lib


def _roundings(n, term):
    """The most roundings a term of a key over n values passes, by running the reference's order
    of additions (distance.rs:3-39) on their counts; a sum of nothing and x is x."""
    def add(a, b):
        return b if a is None else max(a, b) + 1

    lanes = [None] * 8
    for i in range(n // 8 * 8):
        lanes[i % 8] = add(lanes[i % 8], term)
    total = None
    for v in lanes:
        if v is not None:
            total = add(total, v)
    for _ in range(n % 8):
        total = add(total, term)
    return total


def test_ref_roundings_cover_every_width(lib):
    # the bound on the reference's own rounding counts at least as many operations as a term of
    # its sums passes: a difference rounds once and is squared (two), the square once; a product
    # once. ADC sums add m table entries, each a key over dsub values.
    for n in range(1, 1025):
        for term in (3, 1):
            assert lib.ref_roundings(n) >= _roundings(n, term), n
    for dsub in range(1, 65):
        for m in (1, 2, 7, 48):
            entry = _roundings(dsub, 3)
            assert lib.ref_roundings(dsub) + m >= entry + m - 1, (dsub, m)
