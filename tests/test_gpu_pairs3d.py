"""GPU: a run of 3D pairs from one call (bz_yee3d_run2) gives the bits of single steps: without monitors, with one
table (its samples taken by the next pair's launch), with tables of different record steps, with sources in several
tiles, from even and odd step counts, in one run and in pieces."""
import numpy as np
import pytest

import beamz_amd as bz

pytestmark = pytest.mark.gpu

DX = 40e-9


def world(shape, steps, intervals, nsrc):
    nz, ny, nx = shape
    rng = np.random.default_rng(nx + steps)
    d = bz.Design((nx + 1e-6) * DX, (ny + 1e-6) * DX, depth=(nz + 1e-6) * DX, material=bz.Material(1.0),
                  auto_pml=False)
    for q in range(nsrc):
        at = tuple(min(1 + 19 * q, n - 1) * DX for n in (nx, ny, nz))
        d += bz.GaussianSource(position=at, width=DX, signal=np.cos((0.05 + 0.01 * q) * np.arange(steps)))
    mons = []
    for q, interval in enumerate(intervals):
        mons.append(bz.Monitor(design=d, plane_normal="x", plane_position=(nx // 2 + q) * DX, start=((nx // 2 + q) * DX, 0, 0),
                               size=((ny - 1) * DX, (nz - 1) * DX), dft_frequencies=[1.9e14, 2.0e14][: q + 1],
                               record_fields=True, accumulate_power=False, record_interval=interval))
        d += mons[-1]
    eps, sig = 1.0 + 3.0 * rng.random(shape), 2e4 * rng.random(shape)
    sig[:, :, nx // 3:] = 0.0
    t = np.arange(steps) * (0.9 * DX / (bz.LIGHT_SPEED * np.sqrt(3)))
    return bz.FDTD(bz.RegularGrid3D.from_arrays(d, eps, sig, DX, DX), time=t), mons


def run(pairs, pieces, *a):
    sim, mons = world(*a)
    sim.grid.kernel, sim.grid.tb2 = "fused", pairs
    if pieces:
        sim.initialize_simulation(save=False, live=False)
        steps, at = sim.num_steps, 0
        for end in (3, steps // 2, steps):
            sim.grid.run(at, end - at)
            at = end
        r = {k: v.cpu().numpy() for k, v in sim.grid.f.items()}
        for q, plan in enumerate(sim._plans):
            r.update({f"dft{q}": plan.dft.cpu().numpy(), f"series{q}": plan.series.cpu().numpy()})
        return r
    sim.run(live=False, save=False)
    r = {k: np.real(getattr(sim, k)).copy() for k in ("Ex", "Ey", "Ez", "Hx", "Hy", "Hz")}
    for q, m in enumerate(mons):
        r.update({f"dft{q}{k}": np.array(v) for k, v in m.dft.items()})
        r.update({f"series{q}{k}": np.array(v) for k, v in m.fields.items() if len(v)})
    return r


@pytest.mark.parametrize("shape,steps,intervals,nsrc,pieces", [
    ((5, 6, 7), 2, (), 1, False),               # one pair, smaller than a tile, no samples
    ((9, 13, 61), 3, (1,), 1, False),           # one pair and a step; two column tiles
    ((12, 25, 60), 20, (1,), 4, False),         # one table: even record steps in the staging box, odd in the fields
    ((12, 25, 60), 21, (2,), 2, False),         # only first steps of a pair are recorded
    ((12, 25, 60), 21, (3, 1), 4, False),       # two tables, every source box
    ((12, 25, 60), 21, (1,), 2, True),          # one table, taken by the pairs of three calls
    ((12, 25, 60), 21, (2,), 4, True),
    ((12, 25, 60), 21, (5, 1, 2), 2, True)])
def test_pairs_of_one_call_give_the_bits_of_single_steps(hip, shape, steps, intervals, nsrc, pieces):
    a = run(False, pieces, shape, steps, intervals, nsrc)
    b = run(True, pieces, shape, steps, intervals, nsrc)
    assert set(a) == set(b) and len(a) >= 6 + 2 * len(intervals) and np.any(a["Ez"])
    for k in a:
        assert np.array_equal(a[k], b[k]) and (not pieces or np.any(a[k])), k
