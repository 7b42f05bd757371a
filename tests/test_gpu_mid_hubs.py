"""Hubs joined by a repulsive edge in the queued rounds (mid.hip): the cycle test
gives up on them and the round is searched stage by stage, with the same result."""
import os
import re

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TABLE = os.path.join(ROOT, "rama_amd", "tuning", "gfx950.table")


def _two_hubs(arms, seed):
    """Two hubs of `arms` attractive neighbours, each with one more attractive
    neighbour, joined by a repulsive edge, beside an attractive grid whose
    matchings keep the rounds going.  No conflicted cycle."""
    rng = np.random.default_rng(seed)
    h, w = 150, 150
    v = np.arange(h * w).reshape(h, w)
    ii, jj = [v[:, :-1].ravel(), v[:-1].ravel()], [v[:, 1:].ravel(), v[1:].ravel()]
    cc = [rng.uniform(1.0, 2.0, x.size) for x in ii]
    x, y = h * w, h * w + 1
    a = y + 1 + np.arange(arms)
    for hub, arm in ((x, a), (y, a + 2 * arms)):
        ii += [np.full(arms, hub), arm]
        jj += [arm, arm + arms]
        cc += [rng.uniform(0.2, 0.3, arms), rng.uniform(0.5, 1.0, arms) * 0.1]
    ii.append(np.array([x])), jj.append(np.array([y])), cc.append(np.array([-9.0]))
    return (np.concatenate(ii).astype(np.int32), np.concatenate(jj).astype(np.int32),
            np.concatenate(cc).astype(np.float32))


@pytest.mark.parametrize("length,arms", [(5, 3000), (4, 3000), (5, 40), (3, 3000)])
def test_hub_pairs_leave_the_queued_rounds(gpu, monkeypatch, capfd, length, arms):
    i, j, c = _two_hubs(arms, length)
    opts = gpu.options("PD+", verbose=0)
    opts.max_cycle_length_primal = length
    L = gpu.lib()
    got = []
    try:
        for on in (1, 0):
            assert L.rama_tuning_set(b"mid_rounds", 1 << 18, on) == 0
            capfd.readouterr()
            monkeypatch.setenv("RAMA_STAGE_TIMES", "1")
            labels, lb, _, _ = gpu.solve(i, j, c, opts)
            monkeypatch.delenv("RAMA_STAGE_TIMES")
            err = capfd.readouterr().err
            got.append((labels.tolist(), lb, [int(r) for r in re.findall(r"edges, mid, reason (\d+)", err)]))
    finally:
        L.rama_tuning_load(TABLE.encode() if os.path.exists(TABLE) else None)
    assert got[0][:2] == got[1][:2]
    assert got[0][2] and not got[1][2]  # queued rounds ran, and did not with the knob at 0
    # 3000 x 3000 pairs of neighbours: kMidSkew; 40 x 40, or a search of one
    # list's 3000 neighbours in the other: not
    assert (6 in got[0][2]) == (length > 3 and arms > 1000)
