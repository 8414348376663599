"""The byte ranges that the any-k tile GEMV copies read (csrc/gemv_kquant.hip),
from the functions of csrc/load_offsets.h that the kernels call, compiled for the
host: all start on a dword, cover their block and stay inside the operands for
the shapes the dispatch takes."""
from __future__ import annotations

import ctypes
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qgemm-perf-framework-ng_amd", "csrc")
CXX = os.environ.get("CXX", "g++")
pytestmark = pytest.mark.skipif(shutil.which(CXX) is None, reason="needs a host C++ compiler")

SOURCE = r"""
#include "load_offsets.h"
using namespace pfng;

// Weight copies of an n x nsb matrix that break the rules: wave by wave as the
// kernel addresses them, 16 rows from n0 (rows past the matrix repeat the last),
// five 16-byte columns from the copy's start.
extern "C" long bad_iq2_copies(int n, int nsb) {
    const long size = 66L * n * nsb;
    long bad = 0;
    for (int n0 = 0; n0 < n; n0 += 16)
        for (int sb = 0; sb < nsb; ++sb) {
            const long src = (long)(n0 * nsb + sb) * 66 - iq2_copy_back(sb) - 2;
            for (int row = 0; row < 16; ++row) {
                const int r = row < n - n0 ? row : n - n0 - 1;
                const long start = src + (long)r * nsb * 66 + 2 - iq2_copy_odd(sb + r * (nsb & 1));
                const long block = 66L * ((n0 + r) * nsb + sb), at = start + iq2_copy_back(sb) + iq2_copy_odd(sb + r * nsb);
                bad += start % 4 != 0 || start < 0 || start + 80 > size || at != block || block + 66 > start + 80;
            }
        }
    return bad;
}

extern "C" int q4k_half1(int shared_alignment) { return shared_alignment ? kQ4kHalf1Chunk : kQ4kHalf1Block; }
"""


@pytest.fixture(scope="module")
def copies(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("copies") / "copies.so")
    subprocess.run([CXX, "-std=c++17", "-O2", "-shared", "-fPIC", "-Wall", "-I", CSRC, "-x", "c++", "-", "-o", out],
                   input=SOURCE.encode(), check=True, timeout=300)
    lib = ctypes.CDLL(out)
    lib.bad_iq2_copies.restype = ctypes.c_long
    return lib


@pytest.mark.parametrize("n", [1, 2, 3, 16, 17, 31, 33, 50])
@pytest.mark.parametrize("nsb", [8, 9, 10, 11, 21, 43])
def test_iq2_xxs_weight_copies(copies, n, nsb):
    """An even number of blocks, as the dispatch asks; an odd one would read past
    the matrix (kq_tiles_take declines it)."""
    assert (copies.bad_iq2_copies(n, nsb) == 0) == (n * nsb % 2 == 0)


def test_q8_K_copies(copies):
    """Where rows do not share one alignment: H0 is the block's first 144 bytes, H1
    176 bytes (iq2_xxs: bytes 128..271), all from dwords inside the block and
    together covering it. With a shared one a block of index b starts 4 (b % 4)
    bytes past a 16-byte boundary, from which 19 chunks are copied, H1 from chunk 8:
    a row's last block (b % 4 == 3) is left where it ends."""
    h1 = copies.q4k_half1(0)
    assert h1 % 4 == 0 and h1 <= 144 and h1 + 176 == 292 and 128 + 144 <= 292
    h1 = copies.q4k_half1(1)
    assert h1 == 8 * 16 and all((292 * b - 4 * (b % 4)) % 16 == 0 for b in range(8))
    assert -4 * 3 + h1 + 176 == 292
