"""The autotuner's search, with the timing replaced by a formula (no GPU)."""
import json

import pytest

from specter_amd import autotune
from specter_amd.lib import SPX_FP32_MIXED, SPX_FP64


class _Lib:
    """records the overrides in force as spx_tune_line / spx_tune_wall set them"""

    def __init__(self):
        self.clear()

    def clear(self):
        self.line, self.wall = {}, {}

    def spx_tune_clear(self):
        self.clear()
        return 0

    def spx_tune_line(self, n, csize, lines, threads, tables_global):
        self.line[n, csize] = (lines, threads, tables_global)
        return 0

    def spx_tune_wall(self, n, blocks, waves):
        self.wall[n] = (blocks, waves)
        return 0


def _tune(monkeypatch, cost, precision, compiled):
    lib, seen = _Lib(), []

    def time_steps(grid, prec, members):
        n = grid[2]
        line = {cs: lib.line.get((n, cs), (0, 0, -1)) for cs in (16, 8)}
        wall = lib.wall.get(n, (0, 0))
        seen.append((line, wall))
        return cost(line, wall), (16, 8, 0, compiled)

    monkeypatch.setattr(autotune._l, "load_library", lambda: lib)
    monkeypatch.setattr(autotune, "_time_steps", time_steps)
    return autotune.tune_grid(64, 5, precision, 4, log=lambda s: None), seen


def test_register_budget_leaves_the_blocks_to_the_library(monkeypatch):
    """a mixed class faster with three waves per SIMD must not fix the blocks per wave
    of the float64 plans of the same z length"""
    r, _ = _tune(monkeypatch, lambda line, wall: 1.0 - 0.05 * (wall[1] == 3), SPX_FP32_MIXED,
                 {16: True, 8: True})
    assert r["wall"] == [{"n": 89, "blocks_per_wave": 0, "waves_per_simd": 3}]


@pytest.mark.parametrize("compiled", [True, False])
def test_compiled_lines_are_swept_over_lines_only(monkeypatch, compiled):
    """threads and table places belong to a compiled plan: no time is spent on them and
    no noise in them is kept"""
    r, seen = _tune(monkeypatch,
                    lambda line, wall: 1.0 - 0.1 * (line[16][0] == 4) - 0.1 * (line[16][1] == 32),
                    SPX_FP64, {16: compiled, 8: False})
    swept = any(line[16][1:] != (0, -1) for line, _ in seen)
    assert swept != compiled
    assert r["line"] == [{"n": 89, "csize": 16, "lines": 4, "threads": 0 if compiled else 32,
                          "tables_global": -1}]


def test_shipped_choices_leave_the_blocks_to_the_library():
    """the kernel's own share of blocks per wave is the measured one in float64; an entry
    of another share would also move a served run's rounding off a run's on its own"""
    with open(autotune.DEFAULT_PATH) as fh:
        data = json.load(fh)
    assert [e for e in data["wall"] if e["blocks_per_wave"] != 0] == []
