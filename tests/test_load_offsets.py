"""The byte offsets of csrc/load_offsets.h, the functions the kernels call,
compiled for the host and walked over every row, piece and stage of a tile.

q4_0 GEMM staging: a load of a row past the matrix edge, or of a block past its
row in a partial last stage, must lie out of its buffer resource by the lane
offset alone (the range check may or may not count the uniform offset, and
taking it from the size must not wrap); every other load's five dwords must lie
inside its own row."""
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

// Loads of one operand tile that break the rules. rows: the tile's; valid: those
// inside the matrix; step: rows between the pieces of one lane; kb: blocks per
// stage; weight: 18-byte blocks in whole pieces, else 34-byte blocks in halves.
extern "C" long bad_q4_0_loads(int weight, uint32_t rows, uint32_t valid, uint32_t step, uint32_t kb, uint32_t nb) {
    const uint32_t block = weight ? 18 : 34, per_row = weight ? kb : 2 * kb, stages = (nb + kb - 1) / kb;
    const uint64_t size = (uint64_t)valid * nb * block, row_bytes = (uint64_t)nb * block;
    long bad = size >= kPastEnd;
    for (uint32_t s = 0; s < stages; ++s)
        for (uint32_t row = 0; row < rows; ++row)
            for (uint32_t p = 0; p < per_row; ++p) {
                const uint32_t j = weight ? p : p >> 1, lane_row = row % step, above = row - lane_row;
                const bool in_row = s * kb + j < nb;
                const uint32_t past = s == stages - 1 && nb % kb && j >= nb % kb ? kPastEnd : 0;
                const uint32_t piece = weight ? q4_0_weight_piece(lane_row, p, nb) : q4_0_act_piece(lane_row, p, nb);
                const BufferOffset o = q4_0_stage_piece(piece, above * nb * block, s * kb * block, past);
                const uint64_t at = (uint64_t)o.lane + o.uniform;
                if (row < valid && in_row)
                    bad += at % 4 || at < row * row_bytes || at + 20 > (row + 1) * row_bytes || (uint64_t)o.lane + 20 > size;
                else
                    bad += o.lane < size || o.lane > 0xffffffffu - 16;
                bad += o.uniform >= size;
            }
    return bad;
}
"""


@pytest.fixture(scope="module")
def offsets(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("offsets") / "offsets.so")
    subprocess.run([CXX, "-std=c++17", "-O2", "-shared", "-fPIC", "-Wall", "-I", CSRC, "-x", "c++", "-", "-o", out],
                   input=SOURCE.encode(), check=True, timeout=300)
    lib = ctypes.CDLL(out)
    lib.bad_q4_0_loads.restype = ctypes.c_long
    return lib


@pytest.mark.parametrize("weight", [0, 1])
@pytest.mark.parametrize("kb", [4, 8, 16, 32])
@pytest.mark.parametrize("rows", [32, 64, 128])
def test_q4_0_staging(offsets, weight, kb, rows):
    for nb in (4, 8, 12, 36, 68, 128):
        for valid in {1, 2, rows // 2 - 1, rows - 1, rows}:
            for step in (4, 8, 16, 32):
                bad = offsets.bad_q4_0_loads(weight, rows, valid, step, kb, nb)
                assert bad == 0, f"{bad} loads: {valid} of {rows} rows, {nb} blocks, {kb} per stage, step {step}"


@pytest.mark.parametrize("weight", [0, 1])
def test_q4_0_staging_longest_rows(offsets, weight):
    """k = 2^24, the longest row the tiles take: 32-bit offsets do not wrap. (A
    stage of the whole row stands for its first and last blocks.)"""
    nb = (1 << 24) // 32
    for valid in (1, 127, 128):
        assert offsets.bad_q4_0_loads(weight, 128, valid, 16, nb, nb) == 0
