"""The tests of rounds in one launch and queued rounds compare them with the stage
by stage form; here, that their instances do get there and leave for every reason
there is: a search that finds cycles, nothing left to contract, the forest, a
matching of more than six rounds, a row too long for its bucket, a graph small
enough for one launch, and matchings of four to six rounds queued again."""
import re

import pytest

from tests import test_gpu_mid_rounds as mid
from tests import test_gpu_small_rounds as small

pytestmark = pytest.mark.gpu

MORE, CYCLES, DONE, FOREST, MATCHING, SKEW, SMALL = 0, 1, 2, 4, 5, 6, 7


def _reasons(gpu, monkeypatch, capfd, inst, preset):
    capfd.readouterr()
    monkeypatch.setenv("RAMA_STAGE_TIMES", "1")
    gpu.solve(*inst, gpu.options(preset, verbose=0))
    monkeypatch.delenv("RAMA_STAGE_TIMES")
    lines = re.findall(r"edges, (small|mid), reason (\d+), picks (\d+)", capfd.readouterr().err)
    return [(form, int(r)) for form, r, _ in lines], max([int(p) for _, _, p in lines], default=0)


@pytest.mark.parametrize("kind,preset,seed,form,reason,picks", [
    ("hub", "P", 0, "mid", SKEW, 6),
    ("limit", "P", 0, "mid", MATCHING, 6),
    ("limit", "PD+", 1, "mid", CYCLES, 3),
    ("rings", "P", 0, "mid", SMALL, 3),
    ("grid_long", "P", 0, "mid", SMALL, 6),
    ("grid3d", "PD", 0, "mid", FOREST, 3),
    ("sparse", "PD+", 0, "mid", FOREST, 3),
    ("repeats", "PD+", 1, "mid", DONE, 3),
])
def test_queued_rounds_are_reached(gpu, monkeypatch, capfd, kind, preset, seed, form, reason, picks):
    inst = mid._rings(seed) if kind == "rings" else mid._instance(kind, seed)
    got, most = _reasons(gpu, monkeypatch, capfd, inst, preset)
    assert (form, reason) in got and most == picks


@pytest.mark.parametrize("kind,preset,seed,reason", [
    ("star", "P", 77, MORE),
    ("hubs", "PD+", 77, CYCLES),
    ("few", "PD", 77, DONE),
    ("dense", "PD+", 78, DONE),
    ("bits", "PD+", 77, FOREST),
    ("limit", "P", 77, FOREST),
])
def test_rounds_in_one_launch_are_reached(gpu, monkeypatch, capfd, kind, preset, seed, reason):
    got, _ = _reasons(gpu, monkeypatch, capfd, small._instance(kind, seed), preset)
    assert ("small", reason) in got
