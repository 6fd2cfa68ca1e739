"""What DeviceRun.autotune keeps and takes back (CPU: a run with a clock of its own
stands in for the device)."""

import json
from types import SimpleNamespace

import pytest
import torch

from witwin_maxwell_amd.fdtd import native, runtime


class Run(runtime.DeviceRun):
    """A run of ``steps`` steps; passes of several steps where ``passes`` says so."""

    def __init__(self, passes, steps=300, cost=None):
        self.plan = SimpleNamespace(shape=(121, 121, 121), uses_cpml=True, dispersive=False, dft_frequencies=(),
                                    time_steps=steps)
        self.fused, self.step_index, self.clock, self.ran = True, 0, 0.0, []
        self.program, self._planes, self.passes = native.MwProgram(), [], passes
        self.cost = cost or (lambda tiling: 1.0 + sum(tiling))
        self.program.n_points, self._multi = 1, passes[0] > 0

    def tiling(self):
        return (self.program.xchunk, self.program.shell_chunk, self.program.z_tiling)

    def pass_plan(self):
        return self.passes if self.program.z_tiling == 0 else (0, 0, 0)

    def run(self, count):
        count = max(0, count)
        assert self.step_index + count <= self.plan.time_steps
        self.step_index += count
        self.ran.append(count)
        Event.now += count * self.cost(self.tiling())
        return self

    def reset(self):
        self.step_index = 0


class Event:
    now = 0.0

    def __init__(self, **_):
        self.at = None

    def record(self):
        self.at = Event.now

    def synchronize(self):
        pass

    def elapsed_time(self, end):
        return end.at - self.at


@pytest.fixture(autouse=True)
def clock(monkeypatch):
    monkeypatch.setattr(torch.cuda, "Event", Event)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda *a: None)
    monkeypatch.setattr(runtime, "_TUNED", {})
    monkeypatch.delenv("WITWIN_MAXWELL_AMD_TUNE_CACHE", raising=False)


MARCH = (2, 254, 0)


def test_runs_with_and_without_shared_passes_keep_their_own_choice():
    single, several = Run((0, 0, 0)), Run(MARCH)
    assert single.autotune() == (0, 2, 1)  # the fastest of the explicit tilings
    assert several.autotune() == (0, 0, 0)
    other = Run((0, 0, 0))
    assert other.autotune() == (0, 2, 1) and not other.ran, "cached for its own kind"
    again = Run(MARCH)
    assert again.autotune() == (0, 0, 0) and not again.ran
    assert Run((2, 256, 0)).autotune() == (0, 0, 0)


def test_table_entries_of_other_runs_are_not_taken(tmp_path, monkeypatch):
    path = tmp_path / "tuned.json"
    monkeypatch.setenv("WITWIN_MAXWELL_AMD_TUNE_CACHE", str(path))
    key = "single|(121, 121, 121)|1|0|0"
    path.write_text(json.dumps({key: [8, 2, 4]}))  # written for separate launches
    assert Run(MARCH).autotune() == (0, 0, 0)
    assert Run((0, 0, 0)).autotune() == (8, 2, 4)
    runtime._TUNED.clear()
    path.write_text(json.dumps({key: [0, 0, 0]}))  # left by a run with shared passes
    assert Run((0, 0, 0)).autotune() == (0, 2, 1)


@pytest.mark.parametrize("steps", [1, 2, 5, 9, 16, 300])
def test_timings_are_per_step_that_ran(steps):
    run = Run(MARCH, steps=steps)
    run.autotune(trial_steps=12, cache=False)
    if steps > 4:
        assert run.autotune_timings[(0, 0, 0)] == pytest.approx(1.0)
        assert run.autotune_timings[(8, 4, 4)] == pytest.approx(17.0)
