"""q4_0 GEMM tiles: the staging pieces at their edges, bit for bit.

Each tile configuration of csrc/gemm_mfma.hip at one, two, three and more K
stages (an odd last stage is computed outside the loop, prefetched pieces past
the last stage are clamped to it, and blocks past a row's end read zeros) and
with ragged m and n (rows past the edge read zeros). On the inputs of tests/exact_inputs.py every fp32 step is
exact, so the tolerance is zero."""
from __future__ import annotations

import numpy as np
import pytest

from exact_inputs import exact_case
from test_gpu_exact import assert_bits_equal, dev, say

pytestmark = pytest.mark.gpu

# one, two, three and more stages of the 128x128 tiles; then a grid of m and n at k
# that fill the last stage of some tiles and not of others. tests/test_plan.py checks
# that the plan picks every tile here, with odd and even stage counts
CASES = ([(2048, 4096, 128), (2000, 4100, 256), (1921, 4097, 384), (2048, 4096, 640)]
         + [(m, n, k) for m in (9, 33, 100, 200, 333, 700) for n in (100, 1500, 4100) for k in (128, 384, 1152, 2176)]
         + [(40, 4100, 4096), (130, 4033, 4224), (500, 4000, 1664), (1000, 1500, 1280)]
         # 32x32 in 8 K-waves: one partial stage, two, three, three full; 32x64
         + [(20, 100, 896), (20, 100, 1664), (37, 90, 2944), (20, 100, 3072), (20, 100, 1408), (500, 533, 896)]
         # an even (128x128, 128x64, 64x64 in 2 K-waves) and an odd count (64x64)
         + [(500, 10492, 256), (500, 2265, 1408), (500, 1832, 640), (500, 2265, 640)]
         # an even count (64x64 in 2 waves)
         + [(900, 4100, 512)])


# the tiles that fold their sums after every stage (128x64, 64x64 and its two K-waves), which the
# automatic path takes where two stages' sums would be longer than the tile GEMV's
AUTO_CASES = [(100, 8327, 2048), (100, 8327, 2304), (500, 1832, 768), (33, 8327, 1536), (100, 4430, 2304),
              (500, 2265, 512), (500, 2265, 768)]


@pytest.mark.parametrize("m,n,k,auto", [(*c, False) for c in CASES] + [(*c, True) for c in AUTO_CASES],
                         ids=[f"{m}x{n}x{k}" for m, n, k in CASES] + [f"auto-{m}x{n}x{k}" for m, n, k in AUTO_CASES])
def test_staging_bit_exact(hip, torch_gpu, oracle, m, n, k, auto):
    torch = torch_gpu
    say(f"exact q4_0 staging {m}x{n}x{k}")
    _, aq, w, r, _ = exact_case(oracle, 0, m, n, k, seed=m + n + k)
    assert hip.auto_path(0, m, n, k) == hip.PATH_MFMA or not auto
    got = hip.mul_mat(0, dev(torch, w), dev(torch, aq), m, n, k, path=hip.PATH_AUTO if auto else hip.PATH_MFMA)
    torch.cuda.synchronize()
    rows = np.unique(np.r_[0, m - 1, np.random.default_rng(m).choice(m, min(m, 24), replace=False)])
    expect = oracle.matmul(0, w, np.ascontiguousarray(aq[rows]), len(rows), n, k)
    assert_bits_equal(got.cpu().numpy()[rows], expect, f"{m}x{n}x{k} (|a| <= {r})")


@pytest.mark.parametrize("m,n,k", [(33, 70, 640), (200, 1000, 896), (100, 300, 2176), (250, 4000, 384), (9, 40, 1152)])
def test_block_isums_partial_stage(hip, torch_gpu, oracle, m, n, k):
    """Block sums where the last stage is partly past the row's end."""
    torch = torch_gpu
    say(f"block isums q4_0 {m}x{n}x{k}")
    act, w = oracle.create_input(0, m, n, k, seed=5)
    aq = oracle.quantize_q8_0(act)
    got = hip.block_isums(0, dev(torch, w), dev(torch, aq), m, n, k)
    torch.cuda.synchronize()
    assert np.array_equal(got.cpu().numpy(), oracle.isums(0, w, aq, m, n, k))
