"""The K-quant tile GEMV kernels at the k whose rows do not share one alignment
(q4_K k % 1024 != 0, iq2_xxs k % 2048 != 0), bit for bit on the inputs of
tests/exact_inputs.py (every fp32 step exact, so the tolerance is zero): odd
and even super-block counts, fewer and more than the 16 waves, ragged weight
tiles, every chunk count, iq2_xxs with odd and even row counts. The operands
end with their buffers, and an iq2_xxs matrix with an odd number of blocks
(n and k / 256 both odd) takes the other kernels."""
from __future__ import annotations

import numpy as np
import pytest

from exact_inputs import exact_case
from test_gpu_exact import assert_bits_equal, dev, say

pytestmark = pytest.mark.gpu

CASES = ([(1, m, n, k) for m, n, k in [(4, 33, 1280), (16, 64, 1792), (17, 37, 1280), (64, 100, 1536), (5, 17, 2304),
                                       (33, 48, 2816), (65, 20, 3328), (96, 31, 5376), (128, 16, 4352), (100, 40, 11008)]]
         + [(2, m, n, k) for m, n, k in [(5, 34, 2304), (5, 33, 2560), (16, 64, 2816), (17, 37, 2560), (33, 48, 3328),
                                         (65, 20, 5376), (96, 31, 4608), (128, 16, 4352), (100, 40, 11008),
                                         (9, 1, 2304), (40, 33, 2304), (128, 17, 5376)]])


@pytest.mark.parametrize("qtype,m,n,k", CASES, ids=[f"{c[0]}-{c[1]}x{c[2]}x{c[3]}" for c in CASES])
def test_any_k_bit_exact(hip, torch_gpu, oracle, qtype, m, n, k):
    torch = torch_gpu
    say(f"exact any k type={qtype} {m}x{n}x{k}")
    _, aq, w, r, _ = exact_case(oracle, qtype, m, n, k, seed=m + n + k + qtype)
    got = hip.mul_mat(qtype, dev(torch, w), dev(torch, aq), m, n, k)
    torch.cuda.synchronize()
    assert_bits_equal(got.cpu().numpy(), oracle.matmul(qtype, w, aq, m, n, k), f"{m}x{n}x{k} (|a| <= {r})")


# the shapes whose tile the predicted times choose: one round of 128x64 two-slice
# tiles instead of two of 64x64, one-slice tiles at short k, 64x64 instead of 32x32,
# wide outputs of 17..128 rows on the GEMM (q4_K also on whole-K tiles), the q4_K 32x32
# tile whose partials are added in fp64; ragged edges included
PLAN_CASES = [(q, m, n, k) for q in (1, 2)
              for m, n, k in [(333, 4090, 512), (330, 1530, 2048), (600, 4001, 768), (130, 600, 1280),
                              (100, 11000, 256), (37, 14330, 1024), (65, 6100, 2048), (128, 4200, 2304),
                              (40, 6500, 1024), (333, 1363, 1280), (333, 1363, 2048)]]


@pytest.mark.parametrize("qtype,m,n,k", PLAN_CASES, ids=[f"{c[0]}-{c[1]}x{c[2]}x{c[3]}" for c in PLAN_CASES])
def test_planned_tiles_bit_exact(hip, torch_gpu, oracle, qtype, m, n, k):
    torch = torch_gpu
    say(f"exact plan type={qtype} {m}x{n}x{k}")
    _, aq, w, r, _ = exact_case(oracle, qtype, m, n, k, seed=m + n + k + qtype)
    got = hip.mul_mat(qtype, dev(torch, w), dev(torch, aq), m, n, k)
    torch.cuda.synchronize()
    rows = np.unique(np.r_[0, m - 1, np.random.default_rng(m).choice(m, 14, replace=False)])
    expect = oracle.matmul(qtype, w, np.ascontiguousarray(aq[rows]), len(rows), n, k)
    assert_bits_equal(got.cpu().numpy()[rows], expect, f"{m}x{n}x{k} (|a| <= {r})")
