"""Host side of (Hz, Ex, Ey) batches (no GPU: the engine's tables on the CPU, native calls and timers replaced)."""
from types import SimpleNamespace

import numpy as np
import pytest

from beamz_amd import _native as N
from beamz_amd.simulation.batch import FDTDBatch
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
