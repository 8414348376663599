"""q4_0 GEMM tiles: the staging pieces at their edges, bit for bit.

Each tile configuration of csrc/gemm_mfma.hip at one, two, three and more K
stages (an odd last stage is computed outside the loop, and prefetched pieces
past the last stage are clamped to it) and with ragged m and n (rows past the
edge read zeros). On the inputs of tests/exact_inputs.py every fp32 step is
exact, so the tolerance is zero."""
from __future__ import annotations

import numpy as np
import pytest

from exact_inputs import exact_case
from test_gpu_exact import assert_bits_equal, dev, say

pytestmark = pytest.mark.gpu

# (m, n, k): 128x128 tiles (from 512 of them), 64x64 tiles with 8-block
# stages and with 4-block stages, with two K waves, 32x32 tiles
CASES = [(2048, 4096, 128), (2000, 4100, 256), (1921, 4097, 384), (2048, 4096, 640),
         (1000, 1500, 256), (961, 1473, 768), (1000, 1500, 1280),
         (700, 1100, 128), (65, 33, 384), (250, 129, 640),
         (200, 4100, 2560), (129, 4033, 2048),
         (65, 70, 256), (33, 31, 768), (130, 300, 1280), (17, 33, 1024), (31, 95, 3072)]


@pytest.mark.parametrize("m,n,k", CASES, ids=[f"{m}x{n}x{k}" for m, n, k in CASES])
def test_staging_bit_exact(hip, torch_gpu, oracle, m, n, k):
    torch = torch_gpu
    say(f"exact q4_0 staging {m}x{n}x{k}")
    _, aq, w, r, _ = exact_case(oracle, 0, m, n, k, seed=m + n + k)
    got = hip.mul_mat(0, dev(torch, w), dev(torch, aq), m, n, k, path=hip.PATH_MFMA)
    torch.cuda.synchronize()
    rows = np.unique(np.r_[0, m - 1, np.random.default_rng(m).choice(m, min(m, 24), replace=False)])
    expect = oracle.matmul(0, w, np.ascontiguousarray(aq[rows]), len(rows), n, k)
    assert_bits_equal(got.cpu().numpy()[rows], expect, f"{m}x{n}x{k} (|a| <= {r})")
