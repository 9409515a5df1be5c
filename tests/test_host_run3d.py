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
    g.kseg2, g.kseg3, g.calls = 8, 8, []
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


def test_one_pair_goes_without_the_tables_of_a_run(grid):
    """A run of two steps is one launch and one gather per table, and not the set-up of a whole run's tables."""
    grid.add_gather([0, 1], [11, 12], np.arange(400), np.arange(401.0), [1.0], keep_series=False)
    grid.add_gather([2], [13], np.arange(1, 400, 2), np.arange(401.0), [1.0], keep_series=False)
    grid.run(6, 2)
    assert [c[0] for c in grid.calls] == ["bz_yee3d_step2", "bz_gather2", "bz_gather2"]


@pytest.mark.parametrize("n,steps", [(0, 400), (0, 4), (6, 6), (390, 10), (100, 48)])
def test_rows_of_a_run_are_the_recorded_steps(grid, n, steps):
    """The rows handed to the native call, for runs that look steps up and runs that scan the records."""
    records = [np.arange(400), np.arange(2, 400, 5), np.array([5])]
    for rec in records:
        grid.add_gather([0], [11], rec, np.arange(401.0), [1.0], keep_series=False)
    rows = {}

    def call(name, *a):
        assert name == "bz_yee3d_run2"
        for t in range(a[21]):
            rows[a[20][t].comp] = np.ctypeslib.as_array((N.C.c_int * steps).from_address(a[20][t].row)).copy()
    N.call = call
    grid.run(n, steps)
    want = {}
    for p, rec in zip(grid.monitors, records):
        at = {int(s): q for q, s in enumerate(rec)}
        row = [at.get(s, -1) for s in range(n, n + steps)]
        if max(row) >= 0:
            want[p.comp.data_ptr()] = row
    assert {k: list(v) for k, v in rows.items()} == want


def test_the_staging_box_has_a_second_slot_only_for_calls_that_use_it(grid):
    """One slot for single pairs and for several tables (each pair's samples are taken before the next pair); the run
    of pairs with one table, and three-step launches, add the second."""
    grid.add_gather([0, 1], [11, 500], np.arange(40), np.arange(41.0), [1.0], keep_series=False)
    grid.run(0, 2)
    one = grid._stage["buf"].numel()
    box = list(grid._stage["box"])
    assert one == 6 * box[3] * box[4] * box[5]
    grid.run(2, 8)
    assert grid._stage["buf"].numel() == 2 * one
    assert grid.calls[-1][1][18] == grid._stage["buf"].data_ptr() == grid._stage["base"][0]
    grid.tb3 = True
    grid.run(10, 3)
    assert grid.calls[-2][0] == "bz_yee3d_step3" and grid._stage["buf"].numel() == 2 * one
    assert grid.calls[-2][1][19] == grid._stage["buf"].data_ptr() + 4 * one == grid._stage["base2"][0]
    grid.tb3 = False
    grid.add_gather([1], [500], np.arange(0, 40, 2), np.arange(41.0), [1.0], keep_series=False)
    grid.run(13, 8)
    assert grid.calls[-1][0] == "bz_yee3d_run2" and grid.calls[-1][1][21] == 2
    assert grid._stage["buf"].numel() == 6 * int(np.prod(list(grid._stage["box"])[3:]))
