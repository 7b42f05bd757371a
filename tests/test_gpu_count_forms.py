"""The two forms of the 4- and 5-cycle counts, looking entries up in 2-hop sets
and walking lists, and the change from the one to the other within a count, give
the oracle's triangles; the lists take over where sets would resolve a large
share of the entries, in packs and in small counts."""
import re

import numpy as np
import pytest

from rama_amd import instances as I
from tests.instances_small import named

pytestmark = pytest.mark.gpu


def _ring(n, reach, seed, neg=0.4):
    """Every node joined to the `reach` next ones around a ring: many short cycles."""
    rng = np.random.Generator(np.random.PCG64(seed))
    a = np.repeat(np.arange(n), reach)
    b = (a + np.tile(np.arange(1, reach + 1), n)) % n
    c = rng.uniform(0.5, 1.5, size=n * reach) * np.where(rng.random(n * reach) < neg, -1.0, 1.0)
    return np.minimum(a, b).astype(np.int32), np.maximum(a, b).astype(np.int32), c.astype(np.float32)


def _graph(name):
    if name == "ring":  # 13k rep edges of short lists, two mids per expansion
        return _ring(4000, 8, 3)
    if name == "ring_wide":  # lists of 40 entries
        return _ring(1200, 32, 5)
    if name == "ring_dup":
        i, j, c = _ring(3000, 8, 7)
        pick = np.random.Generator(np.random.PCG64(5)).choice(len(i), size=len(i) // 3)
        return tuple(np.concatenate([x, x[pick]]) for x in (i, j, c))
    return named(name)


@pytest.mark.parametrize("name", ["ring", "ring_wide", "ring_dup", "grid96x128_lr", "er3000", "hubs"])
def test_forms_equal_oracle(gpu, oracle, monkeypatch, name):
    i, j, c = _graph(name)
    r, co, v, (rows, cols) = oracle.dcoo_init(i, j, c)
    for max_len in (4, 5):
        for factor in (0.5, 2.0, 30.0, 200.0):
            o = oracle.conflicted_cycles(r, co, v, rows, cols, max_len, factor)
            for form in ("", "sets", "lists"):
                monkeypatch.setenv("RAMA_COUNT_FORM", form)
                g = gpu.conflicted_cycles(r, co, v, rows, cols, max_len, factor)
                assert g[3] == o[3], (max_len, factor, form)
                for x, y in zip(g[:3], o[:3]):
                    assert np.array_equal(x, y), (max_len, factor, form)


@pytest.mark.parametrize("part", ["none", "queue", "list"])
@pytest.mark.parametrize("name", ["ring_dup", "ring_wide", "hubs"])
def test_sets_without_queue_or_list(gpu, oracle, monkeypatch, name, part):
    """What the sets form does where memory for its queue or its list of hubs is
    short: entries resolved as they come, hubs' rep edges unfiltered."""
    i, j, c = _graph(name)
    r, co, v, (rows, cols) = oracle.dcoo_init(i, j, c)
    monkeypatch.setenv("RAMA_COUNT_FORM", "sets")
    monkeypatch.setenv("RAMA_COUNT_QUEUE", part)
    for max_len in (4, 5):
        for factor in (0.5, 30.0):
            o = oracle.conflicted_cycles(r, co, v, rows, cols, max_len, factor)
            g = gpu.conflicted_cycles(r, co, v, rows, cols, max_len, factor)
            assert g[3] == o[3], (max_len, factor)
            for x, y in zip(g[:3], o[:3]):
                assert np.array_equal(x, y), (max_len, factor)


def _counts(capfd, length):
    err = capfd.readouterr().err
    return [(int(a), int(b)) for a, b in re.findall(r"%d-cycle count[^:]*: (\d+) rep edges \((\d+) by sets\)" % length, err)]


def test_lists_take_over_where_many_entries_pass(gpu, oracle, monkeypatch, capfd):
    monkeypatch.setenv("RAMA_CYCLE_STATS", "1")

    def counts(graph, length=5):
        r, co, v, (rows, cols) = oracle.dcoo_init(*graph)
        capfd.readouterr()
        gpu.conflicted_cycles(r, co, v, rows, cols, 5, 400.0)
        return _counts(capfd, length)

    (r, sets), = counts(_graph("ring"))
    assert 8192 < r and 0 < sets < r  # a first chunk by sets
    (r, sets), = counts(_ring(1000, 8, 9))
    assert 0 < r < 8192 and sets == 0  # few rep edges, short lists
    (r, sets), = counts(_graph("ring_wide"), 4)  # its 4-cycles fill the budget
    assert 8192 < r and sets == 0  # long lists, a count that may go on
    (r, sets), = counts(named("grid96x128_lr"))
    assert 8192 < r and sets == r  # few entries pass


def test_packs_walk_lists(gpu, monkeypatch, capfd):
    insts = [I.batch_instance(k, int(n))[:3] for k, n in enumerate(I.batch_sizes(6, 300, 3000, seed=31))]
    opts = gpu.options("PD+", verbose=0)
    ref = [gpu.solve(*x, opts)[:2] for x in insts]
    capfd.readouterr()
    monkeypatch.setenv("RAMA_CYCLE_STATS", "1")
    for form in ("", "sets"):
        monkeypatch.setenv("RAMA_COUNT_FORM", form)
        got = gpu.solve_batch(insts, opts, workers=1)
        err = capfd.readouterr().err
        packs = re.findall(r"count of a pack: (\d+) rep edges \((\d+) by sets\)", err)
        assert packs and all(s == (r if form else "0") for r, s in packs)
        for (la, lba), (lg, lbg) in zip(ref, got):
            assert lba == lbg and np.array_equal(la, lg)
