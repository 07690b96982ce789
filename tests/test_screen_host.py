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
#include <atomic>
#include <cstdlib>
#include <new>
// allocations fail from the nth on, where n is set
static std::atomic<int> left{-1};
void* operator new(std::size_t n) {
    if (left.load() >= 0 && left.fetch_sub(1) <= 0) throw std::bad_alloc();
    return std::malloc(n);
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }
namespace px { int host_threads() { return 4; } }
extern "C" {
// the sum of [0, n) by parallel_for; at most `allocations` of its allocations succeed (-1: all)
int64_t parallel_sum(int64_t n, int allocations) {
    std::atomic<int64_t> sum{0};
    left = allocations;
    px::parallel_for(n, [&](int64_t lo, int64_t hi) {
        for (int64_t i = lo; i < hi; ++i) sum += i;
    });
    left = -1;
    return sum.load();
}
int64_t ref_roundings(int64_t n) { return px::ref_roundings(n); }
int64_t screen_batch(int64_t ds, int64_t most) { return px::screen_batch(ds, most); }
int screen_batch_fits(int64_t nq, int64_t ds) { return px::screen_batch_fits(nq, ds); }
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("screen_host")
    src, out = d / "shim.cpp", d / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-Wl,-Bsymbolic", "-I", CSRC,
                    "-o", str(out), str(src), "-lpthread"], check=True, timeout=120)
    lib = ctypes.CDLL(str(out))
    lib.ref_roundings.restype = ctypes.c_int64
    lib.ref_roundings.argtypes = [ctypes.c_int64]
    lib.parallel_sum.restype = ctypes.c_int64
    lib.parallel_sum.argtypes = [ctypes.c_int64, ctypes.c_int]
    lib.screen_batch.restype = ctypes.c_int64
    for f in (lib.screen_batch, lib.screen_batch_fits):
        f.argtypes = [ctypes.c_int64, ctypes.c_int64]
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


def test_screen_batch_is_what_the_scan_takes(lib):
    # every batch that a screened search is cut into is one the scan's launcher accepts: past
    # 63,500 dims it is fewer than 16,384 queries, past 1.8M none (such searches are not screened)
    seen = set()
    for ds in [128, 384, 1024, 16_384, 63_488, 63_616, 65_536, 233_088, 1_000_064, 1_863_936,
               1_864_192, 1_900_032, 3_000_064, 2 ** 31]:
        b = lib.screen_batch(ds, 16_384)
        seen.add(b)
        assert 0 <= b <= 16_384
        if b:
            assert lib.screen_batch_fits(b, ds)
        if b < 16_384:
            assert not lib.screen_batch_fits(b + 64, ds), (ds, b)
        assert lib.screen_batch(ds, 1) == min(b, 1)
        assert lib.screen_batch(ds, 1000) == min(b, 1000)
    assert 0 in seen and 16_384 in seen and len(seen) > 4
    assert not lib.screen_batch_fits(16_384, 63_616)  # one launch of the whole batch is refused


def test_parallel_for_without_memory_for_threads(lib):
    # a host pass over a caller's data is at the C ABI's entries: where threads cannot be had, for
    # whatever reason, the calling thread does the rest
    for allocations in (-1, 0, 1, 2, 3):
        for n in (0, 1, 3, 4, 1001):
            assert lib.parallel_sum(n, allocations) == n * (n - 1) // 2, (n, allocations)
