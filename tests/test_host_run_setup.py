"""Host set-up of a run by whole arrays against the plain loops it stands for."""
import numpy as np
import pytest

from beamz_amd.simulation.fdtd import record_steps, time_table


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


@pytest.mark.parametrize("dt", [1.7e-17, np.float64(1.7e-17), np.float32(1.7e-17), np.longdouble(1.7) / 10 ** 17, 2,
                                np.int32(2)])
def test_time_table_adds_in_the_type_of_the_step(dt):
    ref, acc = np.empty(5001), 0
    for n in range(5001):
        ref[n] = acc
        acc += dt
    got = time_table(dt, 5000)
    assert got.dtype == np.float64 and np.array_equal(got, ref)
