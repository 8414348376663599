"""Device weight quantizers at the edges of their layout and arithmetic, byte
for byte against the oracle: block counts around the 64 blocks (8 super-blocks)
of a workgroup, q4_0 outputs two bytes off a dword, and the values whose
quotient the q4_K kernel forms by correction steps: quantization ties, ranges
on both sides of the bounds [2^-40, 2^40] of those steps, ranges far below the
offset, infinities and NaN."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_exact import dev, say

pytestmark = pytest.mark.gpu


def expected(oracle, qtype, x):
    y = oracle.quantize_q4_0(x) if qtype == 0 else oracle.quantize_q4_K(x)
    return y.view(np.uint8).reshape(-1)


Q4_0_COUNTS = [(1, 32), (63, 32), (65, 32), (255, 32), (257, 96)]
Q4_K_COUNTS = [(1, 256), (7, 256), (9, 256), (31, 256), (33, 768)]  # outputs 16-byte aligned


@pytest.mark.parametrize("qtype,rows,k,offset", [(0, *c, o) for c in Q4_0_COUNTS for o in (0, 2)]
                         + [(1, *c, 0) for c in Q4_K_COUNTS])
def test_block_counts(hip, torch_gpu, oracle, qtype, rows, k, offset):
    torch = torch_gpu
    say(f"weight quantizer type={qtype} rows={rows} k={k} offset={offset}")
    x = np.random.default_rng(rows + k).standard_normal((rows, k)).astype(np.float32)
    expect = expected(oracle, qtype, x)
    buf = torch.full((expect.size + 64,), 0xA5, dtype=torch.uint8, device="cuda")
    hip.quantize_weights_gpu(qtype, dev(torch, x), out=buf[16 + offset:16 + offset + expect.size])
    torch.cuda.synchronize()
    got = buf.cpu().numpy()
    assert np.array_equal(got[16 + offset:16 + offset + expect.size], expect)
    assert (np.delete(got, np.s_[16 + offset:16 + offset + expect.size]) == 0xA5).all()


def value_rows(k):
    rng = np.random.default_rng(7)
    rows = []
    for step in (1.0, 0.1, 3.0, 1 / 3, 0.7, 1e-3):  # multiples of half a step: ties of x / ls + lm
        rows.append(np.float32(step) * rng.integers(-31, 32, k).astype(np.float32) / 2)
        rows.append(np.float32(step) * (rng.integers(0, 31, k).astype(np.float32) / 2 - np.float32(5.3)))
    for e in (-148, -126, -100, -45, -41, -40, -39, -37, 35, 36, 37, 40, 44, 100, 126):
        rows.append((rng.uniform(-1, 1, k) * 2.0 ** e).astype(np.float32))
    for base in (1.0, -3.0, 1e6, -1e-20, 1e30):  # ranges of a few units in the last place
        rows.append(np.float32(base) * (1 + rng.integers(0, 20, k).astype(np.float32) * np.float32(2.0 ** -23)))
    wide = rng.standard_normal(k).astype(np.float32)
    wide[::7] *= np.float32(1e-30)
    rows.append(wide)
    return np.ascontiguousarray(np.stack(rows).astype(np.float32))


@pytest.mark.parametrize("qtype", [0, 1])
def test_values(hip, torch_gpu, oracle, qtype):
    torch = torch_gpu
    say(f"weight quantizer values type={qtype}")
    x = value_rows(4096)
    got = hip.quantize_weights_gpu(qtype, dev(torch, x)).cpu().numpy()
    expect = expected(oracle, qtype, x).reshape(x.shape[0], -1)
    differs = (got != expect).any(1)
    if qtype == 0:
        # where a scale max / -8 is below 2^-128 its reciprocal overflows, and the
        # conversion of the infinite product to int is the device's, not x86's
        differs &= np.abs(x).reshape(x.shape[0], -1, 32).max(2).min(1) >= 2.0 ** -125
    bad = np.flatnonzero(differs)
    assert bad.size == 0, f"rows {bad} differ"


def test_q4_0_infinite_and_nan(hip, torch_gpu, oracle):
    """Blocks of NaNs, and of NaNs or infinities beside finite values: the scan
    for the largest magnitude passes over NaN, so a block of 32 NaNs keeps the
    initial 0 (scale -0), whether the other blocks of its wave (64 blocks)
    have a tie of magnitudes (an all-zero block does) or not."""
    torch = torch_gpu
    nan, inf = np.float32(np.nan), np.float32(np.inf)
    plain = np.random.default_rng(11).standard_normal((64, 32)).astype(np.float32)
    plain[:, 5] = 9.0  # one largest magnitude per block: no ties
    cases = {"one all-NaN block": np.full((1, 32), nan)}
    for name, rows in {"all-NaN blocks, no tie in the wave": {17: nan, 40: -nan},
                       "an all-NaN block beside a zero block": {17: nan, 40: 0.0}}.items():
        x = plain.copy()
        for r, v in rows.items():
            x[r] = v
        cases[name] = x
    x = plain.copy()
    x[3, 0] = nan  # the first value
    x[4, 5] = nan  # the largest
    x[5, 1:] = nan  # all but one
    x[6] = nan
    x[6, 31] = -2.5
    x[7, 9] = inf
    x[8, 9] = -inf
    x[9, [9, 20]] = inf, -inf
    x[10, [9, 20]] = -inf, inf
    x[11, [9, 20]] = nan, -inf
    cases["NaN and infinities beside finite values"] = x
    for name, x in cases.items():
        say(f"q4_0 inf / nan: {name}")
        got = hip.quantize_weights_gpu(0, dev(torch, x)).cpu().numpy().reshape(-1, 18)
        bad = np.flatnonzero((got != expected(oracle, 0, x).reshape(-1, 18)).any(1))
        assert bad.size == 0, f"{name}: blocks {bad} differ"


def test_q4_K_infinite_and_nan(hip, torch_gpu, oracle):
    """Super-blocks with infinities and NaN, each case in a wave (eight
    super-blocks) of its own, whole super-blocks byte for byte: an infinite value
    makes its sub-block's range infinite, which takes the wave out of the
    correction steps' bounds; a NaN leaves the range finite, so it reaches the
    correction steps (unless all of its sub-block is NaN) and quantizes to 0.
    The reference passes over a NaN that is not its sub-block's first value."""
    torch = torch_gpu
    nan, inf = np.float32(np.nan), np.float32(np.inf)
    plain = np.random.default_rng(3).standard_normal((8, 256)).astype(np.float32)
    places = {"+inf": [(0, 40, inf)], "-inf": [(1, 77, -inf)], "both": [(2, 3, inf), (2, 9, -inf), (5, 200, inf)],
              "NaN": [(0, 33, nan), (3, 1, nan), (3, 255, nan), (6, 130, -nan)],
              "all but one NaN": [(4, i, nan) for i in range(33, 64)],
              "a NaN sub-block": [(4, i, nan) for i in range(32, 64)],
              "NaN beside inf": [(7, 65, nan), (7, 70, inf)]}
    for name, values in places.items():
        x = plain.copy()
        for b, i, v in values:
            x[b, i] = v
        say(f"q4_K inf / nan: {name}")
        got = hip.quantize_weights_gpu(1, dev(torch, x)).cpu().numpy().reshape(8, 144)
        bad = np.flatnonzero((got != expected(oracle, 1, x).reshape(8, 144)).any(1))
        assert bad.size == 0, f"{name}: super-blocks {bad} differ"


def test_q4_K_leading_nan(hip, torch_gpu, oracle):
    """A NaN that is its sub-block's first value makes the reference's range NaN
    (its minimum starts there); the kernel's minimum and maximum pass over it like
    any other, so the bytes are those of the same values with the NaN second."""
    torch = torch_gpu
    say("q4_K leading nan")
    x = np.random.default_rng(4).standard_normal((8, 256)).astype(np.float32)
    x[2, 64] = np.nan
    moved = x.copy()
    moved[2, [64, 65]] = x[2, [65, 64]]
    got = hip.quantize_weights_gpu(1, dev(torch, x)).cpu().numpy().reshape(8, 144)
    expect = expected(oracle, 1, moved).reshape(8, 144).copy()
    # sub-block 2: the low nibbles of qs[32..63], whose first two values change places back
    q = expect[2, 16 + 32:16 + 34]
    expect[2, 16 + 32:16 + 34] = (q & 0xF0) | (q[::-1] & 0x0F)
    assert np.array_equal(got, expect)
