"""The GEMM plans (csrc/gemm_mfma.hip and gemm_kquant.hip, on the CPU): the staging tests reach
every tile, and the automatic path's tiles keep to their rounding limit over
many shapes."""
from __future__ import annotations

import ctypes
import importlib.util
import os

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CUS = 256
# plan index: (rows, columns, blocks per stage, K-waves, stages between folds)
TILES = {0: (128, 128, 4, 1, 0), 1: (128, 64, 8, 1, 2), 2: (128, 64, 8, 1, 1), 3: (64, 64, 16, 2, 2), 4: (64, 64, 16, 2, 1),
         5: (32, 64, 16, 4, 2), 6: (32, 32, 32, 8, 2), 7: (64, 64, 8, 1, 2), 8: (64, 64, 8, 1, 1), 9: (32, 32, 8, 2, 2),
         10: (64, 64, 4, 1, 0)}
WHOLE = 11


class Plan(ctypes.Structure):
    _fields_ = [("config", ctypes.c_int)]


@pytest.fixture(scope="module")
def plan(pkg):
    f = pkg.lib()._ZN4pfng9plan_mfmaEilllib  # pfng::plan_mfma(int, long, long, long, int, bool)
    f.restype = Plan
    f.argtypes = [ctypes.c_int, ctypes.c_int64, ctypes.c_int64, ctypes.c_int64, ctypes.c_int, ctypes.c_bool]
    return lambda m, n, k, automatic: f(0, m, n, k, CUS, automatic).config


def staging_cases():
    spec = importlib.util.spec_from_file_location("staging", os.path.join(HERE, "test_gpu_gemm_staging.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return [(*c, False) for c in mod.CASES] + [(*c, True) for c in mod.AUTO_CASES]


def test_staging_cases_reach_every_tile(plan):
    """Each tile with an even and an odd number of stages above one (the odd last
    stage is computed behind the loop), and, where a stage has more than 4 blocks,
    with a partial last stage (the per-stage folds are planned at k % 256 == 0, so
    those of 8-block stages have none)."""
    seen = {}
    for m, n, k, automatic in staging_cases():
        config = plan(m, n, k, automatic)
        if config != WHOLE:
            blocks, kb = k // 32, TILES[config][2]
            stages = -(-blocks // kb)
            if stages > 1:
                seen.setdefault(config, set()).add("odd" if stages % 2 else "even")
            if blocks % kb:
                seen.setdefault(config, set()).add("partial")
    for config, tile in TILES.items():
        need = {"odd", "even"} | ({"partial"} if tile[2] > 4 and config not in (2, 8) else set())
        assert need <= seen.get(config, set()), f"tile {config} {tile}: {seen.get(config)}"


def chain(n):
    """Roundings of n terms added one after another: partial sums of 1, 2, .. n terms."""
    return n * (n + 1) / 2


def joined(parts):
    """Partial sums added in order: the roundings of the joins."""
    total, out = 0, 0
    for i, p in enumerate(parts):
        total += p
        out += total if i and p else 0
    return out


def tile_rounding(config, nb):
    if config == WHOLE:
        return 4 * chain(nb // 4) + joined([nb // 4] * 4)
    _, _, kb, waves, fold = TILES[config]
    per_wave = [[] for _ in range(waves)]  # blocks of each wave, stage by stage
    for first in range(0, nb, kb):
        for v in range(waves):
            per_wave[v].append(max(0, min(kb // waves, min(nb, first + kb) - first - v * (kb // waves))))
    out = 0
    for stages in per_wave:
        runs = [sum(stages[i:i + fold]) for i in range(0, len(stages), fold)] if fold else [sum(stages)]
        out += sum(map(chain, runs)) + joined(runs)
    return out + joined([sum(s) for s in per_wave])


def test_automatic_tiles_round_no_more_than_the_gemv(pkg, plan):
    """m = 17..128 where the tile GEMV applies: 16 waves, 8-block groups in turn."""
    moved = set()
    for k in [*range(512, 4097, 256), 5120, 6912, 8192, 11008, 14336, 28672]:
        groups = k // 256
        waves = [8 * len(range(v, groups, 16)) for v in range(16)]
        limit = sum(map(chain, waves)) + joined(waves)
        for m in (17, 32, 33, 48, 64, 65, 96, 100, 128):
            if m > 64 and k < 2048:
                continue
            for n in (4097, 5000, 6100, 8192, 10900, 13594, 16640, 20480, 28672, 32000, 65536, 128256):
                if pkg.auto_path(0, m, n, k) != pkg.PATH_MFMA:
                    continue
                config = plan(m, n, k, True)
                moved.add(config)
                assert tile_rounding(config, k // 32) <= 1.03 * limit, (m, n, k, config)
    assert {2, 4, 8} & moved and {1, 3} & moved  # both ways of folding


@pytest.mark.parametrize("qtype,m,n,k,config", [
    (0, 1335, 4488, 128, 0), (0, 1531, 7108, 512, 0), (0, 2048, 14336, 128, 0), (0, 1945, 4367, 640, 10),
    (1, 46, 4161, 256, 3), (1, 17, 20060, 256, 0), (1, 281, 12579, 1280, 0), (1, 142, 17524, 1280, 0),
    (1, 300, 300, 512, 3), (1, 300, 300, 1024, 5)])
def test_plan_takes_the_measured_tile(pkg, qtype, m, n, k, config):
    """Shapes on which the tiles differ by 2 to 45 %, the predicted times by little:
    the plan is the tile measured fastest among those as exact."""
    f = pkg.lib()._ZN4pfng9plan_mfmaEilllib
    f.restype = Plan
    f.argtypes = [ctypes.c_int, ctypes.c_int64, ctypes.c_int64, ctypes.c_int64, ctypes.c_int, ctypes.c_bool]
    assert f(qtype, m, n, k, CUS, True).config == config
