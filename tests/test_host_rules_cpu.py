"""CPU checks of the rules in gx_host.h that the build's host code decides by."""

import ctypes
import os
import subprocess

import pytest

from .conftest import ROOT

SHIM = r"""
#include <cstdlib>
#include <stdexcept>
#include "gx_host.h"
struct Heap {
  void* p = nullptr;
  ~Heap() { free(p); }
  void* ensure(size_t n) { return p ? p : p = malloc(n); }
};
extern "C" {
// A fill that throws at its first `fails` calls: its calls after `gets`
// requests of the buffer, whose last must have succeeded.
int fill_calls(int fails, int gets) {
  gx::FilledOnce<Heap> t;
  int calls = 0, ok = 0;
  for (int i = 0; i < gets; i++) {
    ok = 0;
    try {
      char* p = (char*)t.get(16, [&](void* q) {
        if (calls++ < fails) throw std::runtime_error("launch");
        *(char*)q = 7;
      });
      ok = *p == 7;
    } catch (const std::runtime_error&) {
    }
  }
  return ok ? calls : -1;
}
int record_bytes(int words, int key_bytes, uint64_t n, const uint64_t* top, unsigned lo, unsigned hi) {
  return gx::record_bucket_bytes(words, key_bytes, n, top, lo, hi);
}
int index_bytes(int key_bytes, uint64_t n, const uint64_t* top, unsigned lo, unsigned hi) {
  return gx::index_bucket_bytes(key_bytes, n, top, lo, hi);
}
unsigned walk_cap(uint64_t nodes) { return gx::walk_cap(nodes); }
double fullest(uint64_t n, int bytes, const uint64_t* top, unsigned lo, unsigned hi) {
  return gx::fullest_bucket(n, bytes, top, lo, hi);
}
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("host_rules")
    src, so = str(d / "shim.cpp"), str(d / "shim.so")
    with open(src, "w") as f:
        f.write(SHIM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I",
                    os.path.join(ROOT, "genomix_amd", "csrc"), "-o", so, src], check=True)
    L = ctypes.CDLL(so)
    u64, u64p, u32, i32 = ctypes.c_uint64, ctypes.POINTER(ctypes.c_uint64), ctypes.c_uint, ctypes.c_int
    L.record_bytes.argtypes = [i32, i32, u64, u64p, u32, u32]
    L.index_bytes.argtypes = [i32, u64, u64p, u32, u32]
    L.walk_cap.argtypes = [u64]
    L.fullest.argtypes = [u64, i32, u64p, u32, u32]
    L.fullest.restype = ctypes.c_double
    return L


def _top(counts):
    return (ctypes.c_uint64 * 256)(*counts)


def _canonical(total):
    """Occurrences by top byte as the canonical choice leaves them: falling
    from twice the mean to nothing."""
    return [total * (511 - 2 * t) // 65536 for t in range(256)]


RECORD_CAP = {1: 16384, 2: 8192}  # records a block sorts
INDEX_CAP = 16384 // 2            # nodes a block's table holds


@pytest.mark.parametrize("key_bytes", [8, 14])
@pytest.mark.parametrize("total", [10**7, 10**8, 6 * 10**8, 4 * 10**9, 3 * 10**10])
@pytest.mark.parametrize("ranges", [2, 3, 8, 32, 128])
def test_bucket_bytes_of_key_ranges(rules, key_bytes, total, ranges):
    """Ranges of even size of the top byte: where two-byte buckets are taken,
    the fullest of any range fits a block's LDS, however few of the 65536
    buckets the range covers; a range of few records keeps them."""
    counts = _canonical(total)
    top = _top(counts)
    words = 1 if key_bytes <= 8 else 2
    lo = 0
    while lo < 256:
        hi, n = lo, 0
        while hi < 256 and (hi == lo or n + counts[hi] <= total // ranges):
            n += counts[hi]
            hi += 1
        worst = max(counts[lo:hi]) / 256
        got = rules.record_bytes(words, key_bytes, n, top, lo, hi)
        assert got in (2, 3)
        if got == 2:
            assert worst <= RECORD_CAP[words]
        if worst < RECORD_CAP[words] / 2:
            assert got == 2
        got = rules.index_bytes(key_bytes, n, top, lo, hi)
        if got == 2:
            assert worst <= INDEX_CAP
        if worst < INDEX_CAP / 2:
            assert got == 2
        lo = hi


def test_bucket_bytes_without_counts(rules):
    """One pass over all keys counts no top bytes: twice the mean bucket."""
    none = _top([0] * 256)
    assert rules.fullest(65536 * 100, 2, none, 0, 256) == 200
    assert rules.fullest(65536 * 100, 3, none, 0, 256) == 200 / 256
    assert rules.record_bytes(1, 8, 5 << 26, none, 0, 256) == 2
    assert rules.record_bytes(1, 8, (5 << 26) + 1, none, 0, 256) == 3
    assert rules.record_bytes(2, 14, 1 << 28, none, 0, 256) == 2
    assert rules.record_bytes(2, 14, (1 << 28) + 1, none, 0, 256) == 3
    assert rules.index_bytes(8, 214_000_000, none, 0, 256) == 2
    assert rules.index_bytes(8, 215_000_000, none, 0, 256) == 3
    for n in (0, 1, 1 << 40):  # short keys have no byte below the bucket's
        assert rules.record_bytes(1, 1, n, none, 0, 256) == rules.index_bytes(1, n, none, 0, 256) == 1
        assert rules.record_bytes(1, 3, n, none, 0, 256) == rules.index_bytes(3, n, none, 0, 256) == 2


def test_bucket_bytes_of_an_empty_range(rules):
    top = _top([0] * 128 + [10] * 128)
    assert rules.record_bytes(1, 8, 0, top, 0, 64) == 2
    assert rules.fullest(0, 2, top, 0, 64) == 0


@pytest.mark.parametrize("fails", [0, 1, 3])
def test_buffer_filled_once(rules, fails):
    """A fill that failed is run again by the next request, one that returned
    is not."""
    assert rules.fill_calls(fails, fails + 1) == fails + 1
    assert rules.fill_calls(fails, fails + 4) == fails + 1


def test_walk_cap(rules):
    """Large graphs walk paths of 8192 nodes from both ends; small ones turn to
    the splitters after 1024 nodes a walk."""
    assert [rules.walk_cap(n) for n in (0, 1, 4096 * 1024, 4096 * 1025, 4096 * 4096, 1 << 30)] == [
        1024, 1024, 1024, 1025, 4096, 4096]
