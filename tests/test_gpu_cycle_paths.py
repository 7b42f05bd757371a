"""Every way the cycle search can count and emit gives the oracle's
triangles: the 2-hop tables (5-cycles) and wave-wide sets (4-cycles) against
per-thread counting (RAMA_CYCLE_TABLES=0), and the per-expansion emit
against the queued one (RAMA_EMIT_FORM), on graphs with triangles, hubs,
repeated edges, and budgets that cut the enumeration short."""
import numpy as np
import pytest

from rama_amd import instances as I
from tests.instances_small import named

pytestmark = pytest.mark.gpu

GRAPHS = ["grid96x128_lr", "grid3d_24", "er3000", "er800_dense", "random_dup", "hubs"]
PATHS = [("1", "dense"), ("1", "queue"), ("0", "dense"), ("0", "queue")]


def _contracted(oracle, name, groups):
    i, j, c = named(name)
    r, co, v, dims = oracle.dcoo_init(i, j, c)
    n = max(dims)
    rng = np.random.Generator(np.random.PCG64(7))
    mp = rng.integers(0, max(2, n // groups), size=n).astype(np.int32)
    r2, c2, v2, dims2, _, _ = oracle.contract(r, co, v, mp)
    return r2, c2, v2, dims2


@pytest.mark.parametrize("name", GRAPHS)
@pytest.mark.parametrize("groups", [1, 3])
def test_cycle_paths_equal_oracle(gpu, oracle, monkeypatch, name, groups):
    if groups == 1:
        i, j, c = named(name)
        r, co, v, (rows, cols) = oracle.dcoo_init(i, j, c)
    else:
        r, co, v, (rows, cols) = _contracted(oracle, name, groups)
    for max_len in (4, 5):
        for factor in (2.0, 0.3):
            o = oracle.conflicted_cycles(r, co, v, rows, cols, max_len, factor)
            for tables, form in PATHS:
                monkeypatch.setenv("RAMA_CYCLE_TABLES", tables)
                monkeypatch.setenv("RAMA_EMIT_FORM", form)
                g = gpu.conflicted_cycles(r, co, v, rows, cols, max_len, factor)
                case = (name, groups, max_len, factor, tables, form)
                assert g[3] == o[3], case
                for a, b in zip(g[:3], o[:3]):
                    assert np.array_equal(a, b), case


def test_cycle_paths_batched_equal(gpu, monkeypatch):
    sizes = I.batch_sizes(16, 300, 6000, seed=31)
    insts = [I.batch_instance(k, int(n))[:3] for k, n in enumerate(sizes)]
    opts = gpu.options("PD+", verbose=0)
    ref = gpu.solve_batch(insts, opts, workers=1)
    for tables, form in PATHS:
        monkeypatch.setenv("RAMA_CYCLE_TABLES", tables)
        monkeypatch.setenv("RAMA_EMIT_FORM", form)
        got = gpu.solve_batch(insts, opts, workers=1)
        for (la, lba), (lg, lbg) in zip(ref, got):
            assert lba == lbg, (tables, form)
            assert np.array_equal(la, lg), (tables, form)


@pytest.mark.parametrize("length", [4, 5])
def test_dual_pass_first_cycles_are_longer(gpu, oracle, length):
    """No 3-cycles (nor 4-cycles): the dual pass's later searches take over
    what the fruitless ones before them built."""
    k, n = 300, 300 * length
    v = np.arange(n, dtype=np.int32).reshape(k, length)
    i, j = v.ravel(), np.roll(v, -1, axis=1).ravel()
    rng = np.random.Generator(np.random.PCG64(length))
    c = rng.uniform(0.5, 1.5, size=n).astype(np.float32)
    c[::length] *= -1.0
    r, co, w, (rows, cols) = oracle.dcoo_init(i, j, c)
    for factor in (2.0, 0.5):
        g = gpu.dual_solver(r, co, w, rows, cols, 5, 5, factor, 2)
        o = oracle.dual_solver(r, co, w, rows, cols, 5, 5, factor, 2)
        assert np.array_equal(g[0], o[0]) and np.array_equal(g[1], o[1]) and g[3] == o[3]
        np.testing.assert_allclose(g[2], o[2], rtol=1e-6, atol=1e-6)
        assert abs(g[4] - o[4]) <= 1e-9 * max(1.0, abs(o[4]))
        assert g[4] > np.minimum(w, 0).sum(dtype=np.float64)


def _shared_hubs(seed):
    """Hubs that share hundreds of attractive neighbours (counts past a byte,
    2-hop neighbourhoods past a group's set, lists past a group's lanes) with
    long runs of repulsive edges, beside ordinary ones."""
    rng = np.random.Generator(np.random.PCG64(seed))
    hubs, leaves = 6, 700
    n = hubs + leaves
    e = {}
    for h in range(hubs):
        for x in rng.choice(leaves, size=420, replace=False):
            e[(h, hubs + int(x))] = 1.0
        for x in rng.choice(leaves, size=60, replace=False):
            e.setdefault((h, hubs + int(x)), -1.0)
    for h in range(hubs):
        for g in range(h + 1, hubs):
            e[(h, g)] = -1.0 if (h + g) % 2 else 1.0
    for a, b in rng.integers(hubs, n, size=(900, 2)):
        if a != b:
            e.setdefault((int(min(a, b)), int(max(a, b))), 1.0 if rng.random() < 0.7 else -1.0)
    keys = sorted(e)
    i, j = (np.array(x, dtype=np.int32) for x in zip(*keys))
    c = np.array([e[k] for k in keys]) * rng.uniform(0.5, 1.5, size=len(keys))
    return i, j, c.astype(np.float32)


@pytest.mark.parametrize("repeats", [False, True])
def test_cycle_counts_of_hubs_equal_oracle(gpu, oracle, monkeypatch, repeats):
    i, j, c = _shared_hubs(3)
    if repeats:  # some pairs twice or three times
        pick = np.random.Generator(np.random.PCG64(5)).choice(len(i), size=len(i) // 4)
        i, j, c = (np.concatenate([x, x[pick]]) for x in (i, j, c))
    r, co, v, (rows, cols) = oracle.dcoo_init(i, j, c)
    for max_len in (4, 5):
        for factor in (4.0, 0.4, 30000.0):
            o = oracle.conflicted_cycles(r, co, v, rows, cols, max_len, factor)
            for tables in ("1", "0"):
                monkeypatch.setenv("RAMA_CYCLE_TABLES", tables)
                g = gpu.conflicted_cycles(r, co, v, rows, cols, max_len, factor)
                assert g[3] == o[3], (max_len, factor, tables)
                for a, b in zip(g[:3], o[:3]):
                    assert np.array_equal(a, b), (max_len, factor, tables)


@pytest.mark.parametrize("extra", [0, 20000])
def test_triangles_of_few_and_many_rep_edges(gpu, oracle, monkeypatch, extra):
    """3-cycles on both sides of the 393216 rep edges up to which groups of
    lanes count and write them, with lists of a few, dozens and hundreds of
    entries; rep edges without cycles fill up the count."""
    i, j, c = _shared_hubs(7)
    d, e, f = named("er800_dense")
    n = int(max(i.max(), j.max())) + 1
    m = n + int(max(d.max(), e.max())) + 1
    k = 393216 - int((c < 0).sum()) - int((f < 0).sum()) + extra
    a = np.arange(k, dtype=np.int32)
    i, j = np.concatenate([i, d + n, m + a]), np.concatenate([j, e + n, m + a + 1])
    c = np.concatenate([c, f, np.full(k, -1.0, np.float32)])
    r, co, v, (rows, cols) = oracle.dcoo_init(i, j, c)
    for factor in (2.0, 0.002):
        o = oracle.conflicted_cycles(r, co, v, rows, cols, 3, factor)
        for form in ("dense", "queue"):
            monkeypatch.setenv("RAMA_EMIT_FORM", form)
            g = gpu.conflicted_cycles(r, co, v, rows, cols, 3, factor)
            assert g[3] == o[3], (factor, form)
            for x, y in zip(g[:3], o[:3]):
                assert np.array_equal(x, y), (factor, form)
