"""Message-passing loops replayed from one captured HIP graph against the
same loops launched kernel by kernel (RAMA_MP_GRAPH=0): labels and lower
bounds identical bit for bit, for single solves and the lockstep batch.
Graph solves are repeated with direct solves in between, so every replay
of a fresh capture is checked."""
import numpy as np
import pytest

from rama_amd import instances as I
from tests.instances_small import named

pytestmark = pytest.mark.gpu

CASES = ["grid96x128_lr", "grid3d_24", "er3000", "er800_dense", "random_dup", "hubs"]


@pytest.mark.parametrize("preset", ["PD", "PD+", "D"])
def test_graph_replay_equals_direct(gpu, monkeypatch, preset):
    opts = gpu.options(preset, verbose=0)
    for name in CASES:
        i, j, c = named(name)
        monkeypatch.setenv("RAMA_MP_GRAPH", "0")
        ref = gpu.solve(i, j, c, opts)[:2]
        for rep in range(3):
            monkeypatch.setenv("RAMA_MP_GRAPH", "1")
            lab, lb = gpu.solve(i, j, c, opts)[:2]
            assert lb == ref[1], (name, rep)
            assert np.array_equal(lab, ref[0]), (name, rep)
            monkeypatch.setenv("RAMA_MP_GRAPH", "0")
            lab0, lb0 = gpu.solve(i, j, c, opts)[:2]
            assert lb0 == ref[1] and np.array_equal(lab0, ref[0]), (name, rep)


def test_graph_replay_equals_direct_batched(gpu, monkeypatch):
    sizes = I.batch_sizes(24, 300, 8000, seed=21)
    insts = [I.batch_instance(k, int(n))[:3] for k, n in enumerate(sizes)]
    opts = gpu.options("PD", verbose=0)
    monkeypatch.setenv("RAMA_MP_GRAPH", "0")
    ref = gpu.solve_batch(insts, opts, workers=1)
    for _ in range(2):
        monkeypatch.setenv("RAMA_MP_GRAPH", "1")
        got = gpu.solve_batch(insts, opts, workers=1)
        for (la, lba), (lg, lbg) in zip(ref, got):
            assert lba == lbg
            assert np.array_equal(la, lg)


@pytest.mark.parametrize("count", [1, 90, 682, 683])
@pytest.mark.parametrize("shared", [False, True])
def test_small_loop_equals_launches(gpu, monkeypatch, count, shared):
    """Message passing of up to 2048 triangles and edges in one launch against
    the loop of launches (with the graph), below and above the limit."""
    rng = np.random.Generator(np.random.PCG64(count))
    a = np.arange(count, dtype=np.int32)
    if shared:  # triangles in books of 30 around one repulsive edge
        b, m = 2 * (a // 30), 2 * (count // 30 + 1) + a
        i = np.concatenate([np.unique(b), b, b + 1])
        j = np.concatenate([np.unique(b) + 1, m, m])
        c = np.concatenate([-rng.uniform(1, 9, len(np.unique(b))), rng.uniform(0.1, 1, 2 * count)])
    else:
        i = np.stack([3 * a, 3 * a, 3 * a + 1], 1).ravel()
        j = np.stack([3 * a + 1, 3 * a + 2, 3 * a + 2], 1).ravel()
        c = rng.uniform(0.1, 1.0, 3 * count)
        c[::3] *= -1.0
    order = np.lexsort((j, i))
    i, j, c = i[order].astype(np.int32), j[order].astype(np.int32), c[order].astype(np.float32)
    n = int(j.max()) + 1
    monkeypatch.setenv("RAMA_MP_GRAPH", "1")
    ref = gpu.dual_solver(i, j, c, n, n, 3, 10, 60.0, 3)
    monkeypatch.delenv("RAMA_MP_GRAPH")
    got = gpu.dual_solver(i, j, c, n, n, 3, 10, 60.0, 3)
    assert got[4] == ref[4] and got[3] == ref[3] and got[4] > np.minimum(c, 0).sum(dtype=np.float64)
    for x, y in zip(got[:3], ref[:3]):
        assert np.array_equal(x, y)
