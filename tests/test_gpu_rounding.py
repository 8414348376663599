"""Where the automatic path leaves the tile GEMV for a GEMM tile (m = 17..128 on
wide outputs), its fp32 sums are no less exact than those of the 16 waves that a
GEMV workgroup has: shapes whose fastest tiles add a row's blocks in longer sums
(each of the q4_0 tiles that do not fold, the whole-K tiles, the one-slice
K-quant tile, q4_K's two K-waves), and some whose tile is within the limit. Both errors are taken
from 64 bits on sampled output columns, the waves' in numpy.

The sampled errors' root mean square scatters by less than 2 % (about 8000
outputs); the plan's limit allows 1.5 %."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_exact import say

pytestmark = pytest.mark.gpu

BLOCK = {0: (32, 18), 1: (256, 144), 2: (256, 66)}


def random_weights(torch, qtype, n, k, seed):
    """Random blocks with fp16 scales in [0.5, 2) (q4_K: minima of half the scale)."""
    qk, size = BLOCK[qtype]
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    w = torch.randint(0, 256, (n, k // qk, size), generator=g, device="cuda", dtype=torch.uint8)
    d = (0.5 + 1.5 * torch.rand((n, k // qk, 1), generator=g, device="cuda")).half()
    w[:, :, 0:2] = d.view(torch.uint8)
    if qtype == 1:
        w[:, :, 2:4] = (7.5 * d).view(torch.uint8)  # about the mean of d * q
    return w.reshape(n, -1)


def wave_sums(oracle, qtype, w, aq, m, k, waves=16):
    """The product with the rows of w, in 64 bits from the exact block sums, and
    in fp32 as so many waves add it: blocks in groups of 256 values dealt out in
    turn, one fused multiply-add per block, the waves' partials in wave order."""
    n = w.shape[0]
    s = oracle.isums(qtype, w, aq, m, n, k).astype(np.float64).reshape(m, n, -1, 2 if qtype == 1 else 1)
    blocks = w.reshape(n, -1, BLOCK[qtype][1])
    a = aq.view(np.uint8).reshape(m, blocks.shape[1], -1)

    def scale(x, at, dtype):
        bytes_ = np.dtype(dtype).itemsize
        return np.ascontiguousarray(x[:, :, at:at + bytes_]).view(dtype)[..., 0].astype(np.float64)

    rounded = lambda x: x.astype(np.float32).astype(np.float64)
    d, ad = scale(blocks, 0, np.float16)[None], scale(a, 0, np.float16 if qtype == 0 else np.float32)[:, None]
    # a block's contribution is exactly x * y
    if qtype == 0:
        x, y, exact = d * ad, s[..., 0], d * ad * s[..., 0]
    elif qtype == 1:
        dmin = scale(blocks, 2, np.float16)[None]
        x, y = rounded(rounded(d * s[..., 0]) - dmin * s[..., 1]), ad
        exact = ad * (d * s[..., 0] - dmin * s[..., 1])
    else:
        x, y = rounded(0.125 * d * ad), s[..., 0]
        exact = 0.125 * d * ad * s[..., 0]
    group, total = 256 // BLOCK[qtype][0], None
    for wave in range(waves):
        acc = np.zeros((m, n))
        for b in range(blocks.shape[1]):
            if b // group % waves == wave:
                acc = rounded(acc + x[..., b] * np.broadcast_to(y, s.shape[:3])[..., b])
        total = acc if total is None else rounded(total + acc)
    return exact.sum(-1), total


@pytest.mark.parametrize("qtype,m,n,k", [
    (0, 64, 16640, 11008), (0, 96, 8448, 4352), (0, 65, 10900, 14336), (0, 100, 20480, 4096), (0, 128, 128256, 4096),
    (0, 60, 9342, 1024), (0, 38, 13880, 1536), (0, 45, 6000, 768), (0, 64, 11008, 4096), (0, 37, 11008, 4096),
    (1, 100, 65600, 8192), (1, 100, 11008, 4096), (1, 40, 6500, 1024), (1, 25, 16347, 1280), (2, 90, 90169, 8192), (2, 128, 11008, 4096)])
def test_automatic_path_as_exact_as_16_waves(hip, torch_gpu, oracle, qtype, m, n, k):
    torch = torch_gpu
    say(f"rounding type={qtype} {m}x{n}x{k}")
    w = random_weights(torch, qtype, n, k, seed=m + n + k)
    g = torch.Generator(device="cuda")
    g.manual_seed(1)
    q = hip.quantize_activation(qtype, torch.randn((m, k), generator=g, device="cuda"))
    cols = torch.randperm(n, generator=g, device="cuda")[:max(64, 8192 // m)]
    exact, waves = wave_sums(oracle, qtype, w[cols].cpu().numpy(), q.cpu().numpy(), m, k)
    got = hip.mul_mat(qtype, w, q, m, n, k)[:, cols].double().cpu().numpy()
    error = lambda x: np.sqrt(((x - exact) ** 2).mean() / (exact ** 2).mean())
    say(f"relative error {error(got):.3g}, 16 waves {error(waves):.3g}, path {hip.auto_path(qtype, m, n, k)}")
    assert error(got) <= 1.05 * error(waves)


@pytest.mark.parametrize("qtype,m,n,k", [(1, 20, 9221, 1280), (1, 80, 9597, 2560), (1, 45, 20393, 1792),
                                         (1, 33, 4096, 3328), (2, 20, 9222, 2304), (2, 128, 4096, 3328)])
def test_tiles_at_other_k_as_exact_as_two_slices(hip, torch_gpu, oracle, qtype, m, n, k):
    """At the k that PFNG_PATH_GEMV declines for m > 16 the 16-row tiles stand in
    for GEMM tiles of at most two slices (about 30000 outputs: 1 % scatter)."""
    torch = torch_gpu
    say(f"rounding type={qtype} {m}x{n}x{k}")
    w = random_weights(torch, qtype, n, k, seed=m + n + k)
    g = torch.Generator(device="cuda")
    g.manual_seed(1)
    q = hip.quantize_activation(qtype, torch.randn((m, k), generator=g, device="cuda"))
    cols = torch.randperm(n, generator=g, device="cuda")[:32768 // m]
    exact, slices = wave_sums(oracle, qtype, w[cols].cpu().numpy(), q.cpu().numpy(), m, k, 2)
    got = hip.mul_mat(qtype, w, q, m, n, k)[:, cols].double().cpu().numpy()
    error = lambda x: np.sqrt(((x - exact) ** 2).mean() / (exact ** 2).mean())
    say(f"relative error {error(got):.3g}, two slices {error(slices):.3g}")
    assert error(got) <= 1.02 * error(slices)
