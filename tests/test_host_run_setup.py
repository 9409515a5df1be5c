"""Host set-up of a run by whole arrays against the plain loops it stands for."""
import numpy as np
import pytest

from beamz_amd.simulation.fdtd import record_steps


@pytest.mark.parametrize("every", [1, 3, 0, -2, True, np.int8(3), np.uint8(1), np.uint64(7), np.int64(5), 2.5,
                                   np.float32(1.5)])
@pytest.mark.parametrize("last", [-1, 0, 6, 990, 2.5])
def test_record_steps_are_those_of_the_loop(every, last):
    ref, at = [], last
    for n in range(1000):
        if n - at >= every:
            ref.append(n)
            at = n
    assert list(record_steps(last, every, 1000)) == ref
