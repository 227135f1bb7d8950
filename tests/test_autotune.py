"""The autotuner's cache (CPU; the timed calls are stand-ins): a schedule is
reused only under the version of its meaning it was timed for, and the launches'
own choice is among the candidates."""

import json

import pytest

from plainmp_amd import autotune


class _Cst:
    def __init__(self):
        self.applied = []

    def _dev_set_schedule(self, *s):
        self.applied.append(s)


class _Mv:
    """Fastest with the launch's own choice of block and 8 waves a CU."""

    def __init__(self, cst):
        self.cst, self.calls = cst, 0

    def _dev_check_motions(self, *args):
        self.calls += 1

    def _dev_edge_kernel_ms(self, stream):
        block, waves = self.cst.applied[-1][:2]
        return 1.0 + block + abs(waves - 8)


@pytest.fixture
def tuned(tmp_path, monkeypatch):
    monkeypatch.setattr(autotune, "_device_name", lambda: "card")
    path = str(tmp_path / "cache.json")

    def tune():
        cst = _Cst()
        mv = _Mv(cst)
        schedule, report = autotune.tune_edges(mv, cst, 0, 0, 100, 0, 0, 0, key="job", cache=path)
        return schedule, report, mv.calls, cst.applied[-1]

    return path, tune


def test_schedules_saved_before_the_values_changed_their_meaning(tuned):
    path, tune = tuned
    old = {"block": 256, "waves_per_cu": 32, "kernel_ms": 0.1}
    with open(path, "w") as f:
        json.dump({"card|edges|job|E=100": old, "card|v1|edges|job|E=100": old}, f)
    schedule, report, calls, last = tune()
    assert not report["cached"] and calls > 0
    assert (schedule.block, schedule.waves_per_cu) == (0, 8) == last[:2]
    schedule, report, calls, last = tune()  # its own entry is reused
    assert report["cached"] and calls == 0
    assert (schedule.block, schedule.waves_per_cu) == (0, 8) == last[:2]
    with open(path) as f:
        assert json.load(f)["card|edges|job|E=100"] == old


@pytest.mark.parametrize("candidates", ["EDGE_BLOCKS", "EDGE_WAVES_PER_CU", "EVAL_WHOLE_CHUNKS", "PAIR_SHARES"])
def test_the_launches_own_choice_is_timed(candidates):
    assert 0 in getattr(autotune, candidates)
