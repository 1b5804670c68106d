"""The wait of the LBVH's one-launch sort passes (csrc/pga_lookback.h), on the
CPU: the sum over the tiles before a tile is right whatever words are there,
late or missing, and the wait ends after the looks it is allowed. (Waiting
without a bound, a build whose words another build had cleared held the GPU.)"""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HARNESS = r"""
#include "pga_lookback.h"
// words[k] can be seen from the appear[k]-th idle look on; -1 in *idles: the
// wait went on past any bound
extern "C" uint32_t sum_before(uint32_t tile, uint32_t patience, const uint64_t* words, const uint32_t* appear,
                               const uint32_t* counts, int64_t* idles, uint32_t* counted) {
    *idles = 0;
    *counted = 0;
    try {
        return bvhk::look_back(
            tile, patience, [&](uint32_t k) { return *idles >= (int64_t)appear[k] ? words[k] : 0ull; },
            [&] { if (++*idles > 1000000) throw 0; },
            [&](uint32_t k) { ++*counted; return counts[k]; });
    } catch (int) {
        *idles = -1;
        return 0;
    }
}
"""
COUNT, PREFIX = 1 << 62, 2 << 62
NEVER = 0xFFFFFFFF


@pytest.fixture(scope="module")
def sum_before(tmp_path_factory):
    d = tmp_path_factory.mktemp("lookback")
    src, lib = str(d / "harness.cpp"), str(d / "harness.so")
    with open(src, "w") as f:
        f.write(HARNESS)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror", "-fPIC", "-shared", "-I",
                    os.path.join(ROOT, "operatorgraph_amd", "csrc"), src, "-o", lib], check=True)
    fn = C.CDLL(lib).sum_before
    fn.restype = C.c_uint32

    def call(tile, patience, words, appear, counts):
        idles, counted = C.c_int64(), C.c_uint32()
        w, a, c = (np.ascontiguousarray(x) for x in (words, appear, counts))
        assert w.dtype == np.uint64 and a.dtype == np.uint32 and c.dtype == np.uint32
        s = fn(C.c_uint32(tile), C.c_uint32(patience), C.c_void_p(w.ctypes.data), C.c_void_p(a.ctypes.data),
               C.c_void_p(c.ctypes.data), C.byref(idles), C.byref(counted))
        return s, idles.value, counted.value
    return call


def words_of(counts, prefix):
    """Status words: tile k's count, or where prefix[k] the count up to it."""
    total = np.cumsum(counts, dtype=np.uint64)
    return np.array([(PREFIX | int(total[k])) if prefix[k] else (COUNT | int(counts[k])) for k in range(len(counts))],
                    dtype=np.uint64)


@pytest.mark.parametrize("tile", [0, 1, 2, 7, 8, 9, 16, 17, 245])
@pytest.mark.parametrize("late", ["none", "some", "cleared", "all"])
def test_sum_of_the_tiles_before(sum_before, tile, late):
    rng = np.random.default_rng(tile * 7 + len(late))
    for _ in range(20):
        n = max(tile, 1)
        counts = rng.integers(0, 4097, n).astype(np.uint32)
        prefix = rng.random(n) < rng.choice([0.0, 0.1, 0.9])
        prefix[0] = True
        words = words_of(counts, prefix)
        appear = np.zeros(n, dtype=np.uint32)
        patience = 200
        if late == "some":                        # comes within the looks that are allowed
            appear = rng.integers(0, 100, n).astype(np.uint32)
        elif late == "cleared":                   # some words are gone for good
            appear[rng.random(n) < 0.5] = NEVER
        elif late == "all":
            appear[:] = NEVER
        got, idles, counted = sum_before(tile, patience, words, appear, counts)
        assert got == int(counts[:tile].sum())
        assert 0 <= idles <= patience
        if late in ("none", "some"):
            assert counted == 0                   # nothing is counted that can be waited for
        if late == "all":
            assert counted == tile and idles == (patience if tile else 0)
        # no patience at all: the same sum
        got, idles, _ = sum_before(tile, 0, words, appear, counts)
        assert got == int(counts[:tile].sum()) and idles == 0
