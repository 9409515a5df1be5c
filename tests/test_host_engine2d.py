"""Host side of the 2D engine (no GPU: its tables on the CPU, native calls recorded, not made)."""
from types import SimpleNamespace

import numpy as np
import pytest

from beamz_amd import _native as N
from beamz_amd.simulation.engine import Fused2D, Grid


def grid(pol="Hz", nx=70, ny=40):
    import torch
    return Grid(SimpleNamespace(torch=torch, dev="cpu", stream=None), np.ones((ny, nx)), np.zeros((ny, nx)), 1.0, 1.0,
                0.1, pol=pol)


@pytest.mark.parametrize("shape", [(8, 3, 8), (40, 8, 8), (16, 4, 8), (8, 0, 7)])
def test_shapes_that_do_not_apply_leave_the_one_step_kernel(shape):
    """(K, rows, waves) that no kernel has are refused with (Ez, Hx, Hy) and were never read with (Hz, Ex, Ey)."""
    K, rows, waves = shape
    e = Fused2D([grid()], kstep=K, krows=rows, kwaves=waves)
    assert e.kstep == 0 and not e.pairs
    with pytest.raises(ValueError):
        Fused2D([grid("Ez")], kstep=K, krows=rows, kwaves=waves)
    assert Fused2D([grid()], kstep=-1).kstep == 0 and Fused2D([grid()], kstep=8).kstep == 8
    assert Fused2D([grid()]).kstep and not Fused2D([grid()], krows=3).kstep


@pytest.fixture
def calls(monkeypatch):
    """(entry point, arguments) of every native call; descriptors are not uploaded."""
    made = []
    monkeypatch.setattr(N, "call", lambda name, *a: made.append((name, a)))
    monkeypatch.setattr(Fused2D, "_sync_descs", lambda self, n0, slot0=0: None)
    return made


@pytest.mark.parametrize("pol", ["Ez", "Hz"])
def test_coefficients_are_held_by_engines_that_run_k_steps(calls, pol):
    """An engine that only holds tile lists (the reverse sweep's), or only takes single steps, has no coefficient
    arrays; the first K-step launch allocates and fills them."""
    e = Fused2D([grid(pol)], kstep=8)
    assert e.tilesk is not None and e.coefs is None and e.gcs is None
    e.run(0, 7)
    assert e.coefs is None and not e.descs[0].coef
    e.run(7, 8)
    assert e.descs[0].coef == e.coefs[0].data_ptr() and e.descs[0].gc == e.gcs[0].data_ptr()
    assert [c[0] for c in calls].count("bz_yee2d_coef") == 1


@pytest.mark.parametrize("pol", ["Ez", "Hz"])
@pytest.mark.parametrize("count", [1, 7, 9, 10, 15, 16, 17, 18, 24, 31, 40, 48])
def test_steps_short_of_a_launch_take_one_of_their_own(calls, pol, count):
    """The steps of a run that are fewer than K go in one launch on the same tile list, from two on after whole
    launches and from ten on alone; fewer go one by one. The buffers' parity moves once per launch."""
    e = Fused2D([grid(pol)])
    assert e.kstep == 16 and not e.pairs
    e.run(0, count)
    nl, left = divmod(count, 16)
    single = left if left < (2 if nl else 10) else 0
    made = {n: a for n, a in calls}
    assert ("bz_yee2d_runk_steps" in made) == (count > single)
    if count > single:
        a = made["bz_yee2d_runk_steps"]
        assert (a[0], a[7], a[9], a[10]) == (int(pol == "Hz"), 16, 0, count - single) and "bz_yee2d_coef" in made
    assert made.get("bz_yee2d_hz_run" if pol == "Hz" else "bz_yee2d_run", [0] * 7)[6] == single
    assert e.grids[0]._cur == (nl + (left > single) + single) % 2


def test_pairs_take_the_steps_short_of_a_launch(calls):
    e = Fused2D([grid("Ez")], kstep=12, krows=8, kwaves=8, pairs=True)
    e.run(0, 23)
    assert [n for n, _ in calls] == ["bz_yee2d_coef", "bz_yee2d_runk_steps", "bz_yee2d_run2", "bz_yee2d_run"]
    assert calls[1][1][10] == 12


@pytest.mark.parametrize("points,dense", [((), False), ([(j, 30) for j in range(40)], False),
                                          ([(20, i) for i in range(21)], False), ([(20, i) for i in range(22)], True),
                                          ([(j, i) for j in (20, 21) for i in range(70)], True)])
def test_dense_monitor_points_are_those_past_one_entry_per_lane(points, dense):
    """More than 64 entries (points times components) in the rows of one wave: the workgroup takes the samples."""
    g = grid("Ez")
    if points:
        off = np.array([g.offset(0, j, i) for j, i in points])
        comps = np.repeat(np.arange(3), len(off))
        g.add_gather(comps, np.tile(off, 3), np.arange(8), np.arange(9.0), None)
    e = Fused2D([g], kstep=8, krows=4, kwaves=16)
    assert e.dense == dense


@pytest.mark.parametrize("points,dense", [([(20, i) for i in range(50)], False),
                                          ([(j, i) for j in (20, 30) for i in range(50)], False),
                                          ([(j, i) for j in (20, 21) for i in range(50)], True),
                                          ([(j, i) for j in (4, 8, 20, 30) for i in range(50)], True)])
def test_dense_monitor_points_of_many_regions(monkeypatch, points, dense):
    """More regions than are resident at once: the workgroup takes the samples where a wave has more than 192 entries,
    or a region more than 576 and some wave more than 64."""
    monkeypatch.setattr(Fused2D, "RESIDENT", 0)
    g = grid("Ez")
    off = np.array([g.offset(0, j, i) for j, i in points])
    g.add_gather(np.repeat(np.arange(3), len(off)), np.tile(off, 3), np.arange(8), np.arange(9.0), None)
    assert Fused2D([g], kstep=8, krows=4, kwaves=16).dense == dense
