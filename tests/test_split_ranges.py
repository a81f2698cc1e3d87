"""The tokens that each split covers (kvforge_amd/csrc/kvf_split.hpp, compiled
here for the host) against the same in Python's unbounded integers, over the
whole range of lengths that an int holds: the last split's end, and a chunk
rounded up to whole tiles, may lie past 2^31."""
import ctypes
import os
import random
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TILE = 32
LAST = 2 ** 31 - 1

SOURCE = r"""
#include "kvf_split.hpp"
using namespace kvf::gfx950;
extern "C" {
uint32_t chunk_of(int len, int splits, int whole) { return split_chunk(len, splits, whole != 0); }
void range_of(int len, uint32_t chunk, int split, int *out) {
  const TokenRange t = split_range(len, chunk, split);
  out[0] = t.t0;
  out[1] = t.t1;
}
int tiles(int len) { return tiles_of(len); }
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("split")
    (d / "split.cpp").write_text(SOURCE)
    so = str(d / "split.so")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-fsanitize=undefined", "-fno-sanitize-recover",
                    "-shared", "-fPIC", "-I" + os.path.join(ROOT, "kvforge_amd", "csrc"), "-o", so,
                    str(d / "split.cpp")], check=True)
    out = ctypes.CDLL(so)
    out.chunk_of.restype = ctypes.c_uint32
    out.range_of.argtypes = [ctypes.c_int, ctypes.c_uint32, ctypes.c_int, ctypes.POINTER(ctypes.c_int)]
    return out


def check(lib, n, splits, whole, which):
    per = -(-n // splits)
    chunk = -(-per // TILE) * TILE if whole else per
    assert lib.chunk_of(n, splits, int(whole)) == chunk, (n, splits, whole)
    got = (ctypes.c_int * 2)()
    for s in which:
        lib.range_of(n, chunk, s, got)
        assert (got[0], got[1]) == (min(n, s * chunk), min(n, (s + 1) * chunk)), (n, splits, whole, s)


@pytest.mark.parametrize("whole", [False, True])
def test_every_split_of_short_lengths(lib, whole):
    for n in list(range(0, 70)) + [127, 128, 129, 1000, 1003, 4093]:
        for splits in (1, 2, 3, 7, 8, 31, 32, 33, 64, 200):
            check(lib, n, splits, whole, range(splits))


@pytest.mark.parametrize("whole", [False, True])
def test_lengths_up_to_the_last_int(lib, whole):
    rng = random.Random(1)
    for splits in (1, 2, 3, 8, 64, 97, 1000, 65535):
        near = {LAST - k for k in (0, 1, 26, 27, 30, 31, 32, 33, 250, 251, 100)}
        near |= {LAST - rng.randrange(40 * splits) for _ in range(40)} | {rng.randrange(1, LAST) for _ in range(40)}
        for n in near:
            some = {0, 1, splits // 2, splits - 2, splits - 1} | {rng.randrange(splits) for _ in range(4)}
            check(lib, n, splits, whole, sorted(s for s in some if 0 <= s < splits))


def test_tiles(lib):
    for n in (0, 1, 31, 32, 33, 1003, LAST - 32, LAST - 31, LAST - 1, LAST):
        assert lib.tiles(n) == -(-n // TILE)
