"""Which instances leave a lockstep pack for a worker before their forest phase:
those whose rounds the worker runs in one launch, and only of a pack with few
slots per worker.  Read off the rounds the workers print."""
import re

import numpy as np
import pytest

from tests.instances_small import random_graph

pytestmark = pytest.mark.gpu


def _solves(err):
    """Per solve that a worker finished: its rounds' lines, first word after the sizes."""
    out, cur = [], []
    for line in err.splitlines():
        m = re.match(r"rounds? [\d.]+: \d+ edges, (\w+),", line)
        if m:
            cur.append(m.group(1))
        elif line.startswith("solve: "):
            out.append(cur)
            cur = []
    return out


def _batch(gpu, monkeypatch, capfd, insts, preset, workers):
    opts = gpu.options(preset, verbose=0)
    ref = [gpu.solve(*x, opts)[:2] for x in insts]
    capfd.readouterr()
    monkeypatch.setenv("RAMA_STAGE_TIMES", "1")
    got = gpu.solve_batch(insts, opts, workers=workers)
    monkeypatch.delenv("RAMA_STAGE_TIMES")
    for (la, lba), (lg, lbg) in zip(ref, got):
        assert lba == lbg and np.array_equal(la, lg)
    return _solves(capfd.readouterr().err)


@pytest.mark.parametrize("preset", ["P", "PD"])
def test_many_small_instances_stay(gpu, monkeypatch, capfd, preset):
    insts = [random_graph(600, 1900, seed=300 + k, neg_frac=0.3) for k in range(40)]
    solves = _batch(gpu, monkeypatch, capfd, insts, preset, 1)
    # of 40 slots and one worker, only the last 8 may leave while they match
    assert sum("small" in s for s in solves) <= 8
    solves = _batch(gpu, monkeypatch, capfd, insts[:4], preset, 1)
    assert any("small" in s for s in solves)


@pytest.mark.parametrize("preset", ["PD", "PD+"])
def test_leaves_only_for_one_launch(gpu, monkeypatch, capfd, preset):
    # about 2000 nodes after the first contraction: too many for the cycle
    # test of PD+ in one launch, few enough for that of PD
    insts = [random_graph(3000, 4600, seed=400 + k, neg_frac=0.2) for k in range(4)]
    solves = _batch(gpu, monkeypatch, capfd, insts, preset, 1)
    assert all(s[0] in ("small", "forest") for s in solves if s)
