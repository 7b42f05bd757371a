"""Rounds queued without read-backs (mid.hip) against the same rounds stage by
stage: labels and bounds bit for bit, or the same error.  Graphs around the
limits of the queued form: 2^18 edges, few and many nodes, a row bucket too
large for LDS (a hub), matchings of more than three rounds, ties."""
import os

import numpy as np
import pytest

from rama_amd import instances
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
    if kind == "grid_long":
        return instances.grid2d_voronoi(H=97, W=211, n_seeds=20, seed=seed)[:3]
    if kind == "grid3d":
        return instances.grid3d_voronoi(D=41, n_seeds=190, seed=seed)[:3]
    if kind == "limit":  # contracted graphs on both sides of 2^18 edges
        return random_graph(90000 + 20000 * seed, 290000, seed=seed, neg_frac=0.2)
    if kind == "sparse":  # many nodes, long runs of isolated ids
        return random_graph(200000, 60000, seed=seed, neg_frac=0.1)
    if kind == "dense":
        return random_graph(420, 60000, seed=seed, neg_frac=0.5)
    if kind == "hub":  # one row of 20000 entries
        i, j, c = random_graph(20001, 30000, seed=seed)
        k = np.arange(1, 20001, dtype=np.int32)
        w = np.random.default_rng(seed).normal(0.1, 1.0, len(k)).astype(np.float32)
        keep = (np.minimum(i, j) > 0)
        return (np.concatenate([i[keep], np.zeros_like(k)]), np.concatenate([j[keep], k]), np.concatenate([c[keep], w]))
    if kind == "hubs":
        return hub_graph(9000, 20, 600, seed=seed)
    if kind == "repeats":
        return random_graph(9000, 30000, seed=seed, neg_frac=0.2, dup=True)
    i, j, c = random_graph(12000, 40000, seed=seed)  # ties
    return i, j, np.round(c).astype(np.float32)


@pytest.mark.parametrize("preset", ["P", "PD"])
@pytest.mark.parametrize("kind", ["grid_long", "grid3d", "limit", "sparse", "dense", "hub", "hubs", "repeats", "ties"])
def test_queued_equals_stages(gpu, table, kind, preset):
    for seed in range(2):
        i, j, c = _instance(kind, seed)
        opts = gpu.options(preset, verbose=0)
        got = []
        for on in (1, 0):
            assert table.rama_tuning_set(b"mid_rounds", 1 << 18, on) == 0
            assert table.rama_tuning_set(b"small_rounds", 4096, on and seed) == 0
            try:
                labels, lb, _, _ = gpu.solve(i, j, c, opts)
                got.append((labels.tolist(), lb))
            except gpu.RamaError as e:
                got.append(str(e))
        assert got[0] == got[1], "kind %s seed %d" % (kind, seed)


def _rings(seed):
    """Attractive rings of 9 to 40 nodes with one repulsive edge, joined to
    two hubs: contraction shortens the conflicted cycles round by round."""
    rng = np.random.default_rng(seed)
    i, j, c = [], [], []
    base = 2
    for length in rng.integers(9, 41, size=500):
        v = base + np.arange(length)
        w = rng.uniform(0.1, 1.0, size=length)
        w[0] *= -1.0
        i.append(v), j.append(np.roll(v, -1)), c.append(w)
        hub = rng.integers(0, 2, size=2)
        i.append(hub), j.append(rng.choice(v, 2, replace=False)), c.append(rng.normal(-0.2, 0.3, size=2))
        base += length
    i, j = np.concatenate(i), np.concatenate(j)
    perm = rng.permutation(base)  # ids in no order
    i, j = perm[i], perm[j]
    return np.minimum(i, j).astype(np.int32), np.maximum(i, j).astype(np.int32), np.concatenate(c).astype(np.float32)


@pytest.mark.parametrize("length", [3, 4, 5])
@pytest.mark.parametrize("kind", ["rings", "grid_long", "grid3d", "limit", "sparse", "dense", "hub", "hubs", "ties"])
def test_queued_longer_cycles(gpu, table, kind, length):
    for seed in range(2):
        i, j, c = _rings(seed) if kind == "rings" else _instance(kind, seed)
        opts = gpu.options("PD+", verbose=0)
        opts.max_cycle_length_primal = length
        got = []
        for on in (1, 0):
            assert table.rama_tuning_set(b"mid_rounds", 1 << 18, on) == 0
            assert table.rama_tuning_set(b"small_rounds", 4096, on and seed) == 0
            try:
                labels, lb, _, _ = gpu.solve(i, j, c, opts)
                got.append((labels.tolist(), lb))
            except gpu.RamaError as e:
                got.append(str(e))
        assert got[0] == got[1], "kind %s seed %d" % (kind, seed)
