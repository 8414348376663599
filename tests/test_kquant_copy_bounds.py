"""The byte ranges that the any-k tile GEMV copies read (csrc/gemv_kquant.hip),
from the rules the kernels state: all start on a dword and stay inside the
operands for the shapes the dispatch takes."""
from __future__ import annotations

import pytest


@pytest.mark.parametrize("n", [1, 2, 3, 16, 17])
@pytest.mark.parametrize("nsb", [8, 9, 10, 11, 21, 43])
def test_iq2_xxs_weight_copies(n, nsb):
    """80 bytes from a block's start, less 2 where its index is odd and 12 where
    it is not its row's first."""
    size = 66 * n * nsb
    for r in range(n):
        for s in range(nsb):
            block = 66 * (r * nsb + s)
            start = block - (12 if s else 0) - 2 * ((r * nsb + s) & 1)
            assert start % 4 == 0 and start >= 0 and start <= block and block + 66 <= start + 80
            if n * nsb % 2 == 0:
                assert start + 80 <= size


@pytest.mark.parametrize("m", [1, 3])
@pytest.mark.parametrize("nsb", [5, 6, 7, 43])
def test_q8_K_copies(m, nsb):
    """H0: the block's first 144 bytes (iq2_xxs H1: bytes 128..271, q4_K H1 its
    last 176)."""
    size = 292 * m * nsb
    for b in range(m * nsb):
        for start, length in [(0, 144), (128, 144), (116, 176)]:
            at = 292 * b + start
            assert at % 4 == 0 and at + length <= size
            assert start + length <= 292
