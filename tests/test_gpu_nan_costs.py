"""Costs that are not a number, which the entry points take: a graph's rounds in
one launch, queued, in a pack or left to a worker give what they give stage by
stage."""
import os

import numpy as np
import pytest

from tests.instances_small import random_graph

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TABLE = os.path.join(ROOT, "rama_amd", "tuning", "gfx950.table")


@pytest.fixture
def table(gpu):
    L = gpu.lib()
    yield L
    L.rama_tuning_load(TABLE.encode() if os.path.exists(TABLE) else None)


def _with_nan(n, m, share, seed):
    i, j, c = random_graph(n, m, seed=seed, neg_frac=0.2)
    c[np.random.default_rng(seed).random(len(c)) < share] = np.nan
    return i, j, c


def _knob(table, on, *names):
    for name, size in (("small_rounds", 4096), ("mid_rounds", 1 << 18)):
        assert table.rama_tuning_set(name.encode(), size, int(on and name in names)) == 0


@pytest.mark.parametrize("preset", ["P", "PD", "PD+"])
@pytest.mark.parametrize("path,n,m", [("small_rounds", 700, 2500), ("small_rounds", 2500, 3500),
                                      ("mid_rounds", 9000, 30000), ("mid_rounds", 20000, 45000)])
def test_rounds_equal_stages(gpu, table, path, n, m, preset):
    for seed in range(4):
        for share in (0.002, 0.1):
            i, j, c = _with_nan(n, m, share, 50 + seed)
            got = []
            for on in (1, 0):
                _knob(table, on, path)
                labels, lb, _, _ = gpu.solve(i, j, c, gpu.options(preset, verbose=0))
                got.append((labels.tolist(), np.float64(lb).tobytes()))
            assert got[0] == got[1], (seed, share)


@pytest.mark.parametrize("preset", ["P", "PD"])
def test_packs_equal_packs_without_leaving(gpu, table, preset):
    insts = [_with_nan(700, 2500, 0.02 if k % 2 else 0.0, 80 + k) for k in range(8)]
    got = []
    for on in (1, 0):
        _knob(table, on, "small_rounds")
        out = gpu.solve_batch(insts, gpu.options(preset, verbose=0))
        got.append([(lab.tolist(), np.float64(lb).tobytes()) for lab, lb in out])
    assert got[0] == got[1]
