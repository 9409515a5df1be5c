"""Host side of 3D runs (no GPU: the native calls are recorded, not made)."""
from types import SimpleNamespace

import numpy as np
import pytest

from beamz_amd import _native as N
from beamz_amd.simulation.engine import Grid


@pytest.fixture
def grid(monkeypatch):
    """A small 3D grid on the CPU; grid.calls holds (entry point, arguments) of every native call."""
    import torch
    g = Grid(SimpleNamespace(torch=torch, dev="cpu", stream=None), np.ones((8, 9, 10)), np.zeros((8, 9, 10)), 1.0, 1.0, 0.1,
             1.0)
    g.kseg2, g.calls = 8, []
    monkeypatch.setattr(N, "call", lambda name, *a: g.calls.append((name, a)))
    return g


def steps_done(g):
    done = {"bz_yee3d_step": lambda a: 1, "bz_yee3d_step2": lambda a: 2, "bz_yee3d_run2": lambda a: 2 * a[17]}
    return sum(done[name](a) for name, a in g.calls if name in done)


@pytest.mark.parametrize("lengths,steps", [((7,), 6), ((6, 10), 6), ((10, 7), 6), ((3, 9), 2), ((1,), 0), ((0, 4), 0)])
def test_a_run_past_a_source_signal_stops_where_it_ends(grid, lengths, steps):
    """Every step that all sources have samples for runs (in pairs), then the missing sample raises IndexError."""
    for q, n in enumerate(lengths):
        grid.add_point_source("Ez", np.array([[2, 3, 2 + q]]), np.ones(1), None, np.arange(n, dtype=float))
    with pytest.raises(IndexError):
        grid.run(0, 10)
    assert steps_done(grid) == steps


def test_runs_within_the_signals_take_every_step(grid):
    for q, n in enumerate((12, 10)):
        grid.add_point_source("Ez", np.array([[2, 3, 2 + q]]), np.ones(1), None, np.arange(n, dtype=float))
    grid.run(0, 10)
    assert steps_done(grid) == 10 and [c[0] for c in grid.calls] == ["bz_yee3d_run2"]
