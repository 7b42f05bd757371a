"""Rounds of a small graph in one launch (small.hip) against the same rounds
stage by stage: labels and bounds bit for bit, or the same error.  Sizes sit
at the edges of the one-launch form: 4096 edges and nodes, the bit matrix of
the 4- and 5-cycle test (about 800 nodes), few edges, dense graphs, hubs."""
import os

import numpy as np
import pytest

from tests.instances_small import hub_graph, random_graph

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TABLE = os.path.join(ROOT, "rama_amd", "tuning", "gfx950.table")


@pytest.fixture
def table(gpu):
    L = gpu.lib()
    yield L
    L.rama_tuning_load(TABLE.encode() if os.path.exists(TABLE) else None)


def _instance(kind, seed):
    if kind == "few":
        return random_graph(6, 5, seed=seed)
    if kind == "star":
        n = 3000
        c = np.random.default_rng(seed).normal(0.2, 1.0, n - 1).astype(np.float32)
        return np.zeros(n - 1, np.int32), np.arange(1, n, dtype=np.int32), c
    if kind == "dense":  # 90 nodes: 4005 pairs at most
        return random_graph(90, 4000, seed=seed, neg_frac=0.5)
    if kind == "limit":  # first contraction on both sides of 4096 edges
        return random_graph(3000 + 40 * (seed % 5), 4800 + 60 * (seed % 5), seed=seed, neg_frac=0.3)
    if kind == "nodes":  # more than 4096 nodes, sparse
        return random_graph(5200 + 300 * (seed % 4), 4400, seed=seed, neg_frac=0.1)
    if kind == "bits":  # contracted graphs around 800 nodes
        return random_graph(1000 + 60 * (seed % 5), 1700, seed=seed, neg_frac=0.15)
    if kind == "repeats":
        return random_graph(400, 1500, seed=seed, dup=True)
    if kind == "ties":  # few distinct costs
        i, j, c = random_graph(700, 2400, seed=seed)
        return i, j, np.round(c).astype(np.float32)
    return hub_graph(900, 6, 150, seed=seed)


@pytest.mark.parametrize("preset", ["P", "PD", "PD+"])
@pytest.mark.parametrize("kind", ["few", "star", "dense", "limit", "nodes", "bits", "repeats", "ties", "hubs"])
def test_one_launch_equals_stages(gpu, table, kind, preset):
    for seed in range(4):
        i, j, c = _instance(kind, 77 + seed)
        opts = gpu.options(preset, verbose=0)
        got = []
        for on in (1, 0):
            assert table.rama_tuning_set(b"small_rounds", 4096, on) == 0
            try:
                labels, lb, _, _ = gpu.solve(i, j, c, opts)
                got.append((labels.tolist(), lb))
            except gpu.RamaError as e:
                got.append(str(e))
        assert got[0] == got[1], "kind %s seed %d" % (kind, seed)
