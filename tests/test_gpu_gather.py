"""Running aggregates of the recorded pressure (KW_REC_P_AGG), whichever kernel gathers a step.

A block of steps gathers in the column passes of the steps after the first and, for the
last one, in a kernel that also advances the step counter while every sensor has a lane of
one workgroup (256), in two launches beyond; with millions of sensors every step has a
launch of its own.  The maximum, minimum and sum of squares are
read and written again every step, so a step gathered twice, or not at all, shows.
"""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _plan(shape, nt):
    from kwave_amd.data import Vector
    from kwave_amd.kgrid import kWaveGrid
    from kwave_amd.kmedium import kWaveMedium
    from kwave_amd.ksensor import kSensor
    from kwave_amd.ksource import kSource
    from kwave_amd.solvers.plan import DevicePlan
    from kwave_amd.solvers.setup import build_instance

    rng = np.random.default_rng(3)
    kg = kWaveGrid(Vector(list(shape)), Vector([1e-4] * len(shape)))
    kg.setTime(nt, 0.3e-4 / 1700.0)
    src = kSource()
    src.p0 = 1e5 * rng.random(shape)
    sen = kSensor(np.ones(shape, dtype=bool))
    sen.record = ["p"]
    med = kWaveMedium(sound_speed=1500.0 + 200.0 * rng.random(shape), density=1000.0)
    return DevicePlan([build_instance(kg, med, src, sen, pml_size=(3,) * len(shape), pml_alpha=(2.0,) * len(shape))])


def _check(shape, sensors, nt, start, monkeypatch):
    from kwave_amd import _abi

    idx = np.sort(np.random.default_rng(sensors).choice(int(np.prod(shape)), sensors, replace=False)).astype(np.int64)

    def records(steps):
        pl = _plan(shape, nt)
        _abi.check(_abi.lib().kw_plan_set_sensor(pl._h, 0, sensors, 1, idx.ctypes.data_as(C.POINTER(C.c_int64)), None, start,
                                                 _abi.REC_P | _abi.REC_P_AGG))
        pl.reset()
        left = nt - pl.step_index(0)
        while left > 0:
            pl.run(min(steps, left))
            left -= steps
        p, agg = pl.read(0, _abi.F_REC_P).reshape(nt - start, sensors), pl.read(0, _abi.F_AGG_P).reshape(3, sensors)
        pl.close()
        return p, agg

    runs = [records(nt), records(1), records(11)]
    monkeypatch.setenv("KW_NO_GRAPH", "1")
    runs.append(records(nt))
    for p, agg in runs:
        assert np.array_equal(p, runs[0][0]) and np.abs(p).max() > 0
        assert np.array_equal(agg[0], p.max(axis=0)) and np.array_equal(agg[1], p.min(axis=0))
        # nt - start squares and additions in FP32, each rounded by at most 2^-24 of the sum
        np.testing.assert_allclose(agg[2], (p.astype(np.float64) ** 2).sum(axis=0), rtol=2 * (nt - start) * 2.0 ** -24)


@pytest.mark.parametrize("shape", [(70, 66), (128, 64), (20, 18, 16), (32, 16, 24)])
@pytest.mark.parametrize("sensors", [1, 255, 256, 257, 4500])
def test_aggregates_follow_the_recorded_series(shape, sensors, monkeypatch):
    _check(shape, sensors, 30, 5, monkeypatch)


@pytest.mark.parametrize("shape,sensors", [((160, 160, 120), 3000000), ((160, 160, 120), 3000001), ((150, 161, 125), 3018750)])
def test_aggregates_of_very_many_sensors(shape, sensors, monkeypatch):
    """Around the number from which every step of a block gathers in a kernel of its own."""
    _check(shape, sensors, 14, 2, monkeypatch)
