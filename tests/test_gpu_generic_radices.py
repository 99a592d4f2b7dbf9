"""The run-time radix plans of the generic-length family (csrc/kw_generic.hip).

Every butterfly from 2 to 16, direct stages of larger primes (one, two, and in front of
butterflies), the longest lines, and the routes whose lines do not fit LDS together.

Tolerance of a forward and inverse transform: 2e-6 (the family's bar), plus the random
walk of a direct stage's sums, (p - 1) / 2 terms of unit-roundoff 6e-8 each way:
2 * 6e-8 * sqrt(p).
"""
import copy

import numpy as np
import pytest

from test_gpu_fft import _ref, _rel

pytestmark = pytest.mark.gpu

LENGTHS = {6: 3, 9: 3, 10: 5, 11: 11, 12: 3, 13: 13, 14: 7, 15: 5, 22: 11, 26: 13, 90: 5, 108: 3, 143: 13, 210: 7, 17: 17, 34: 17,
           289: 17, 323: 19, 291: 97, 582: 97, 1021: 1021, 2310: 11, 2916: 3, 3003: 13, 4093: 4093, 4095: 13}


@pytest.mark.parametrize("n", sorted(LENGTHS))
@pytest.mark.parametrize("along", [0, 1])
def test_every_radix(n, along):
    from kwave_amd import _abi

    shape = (n, 10) if along == 0 else (7, n)  # the strided and the contiguous axis (odd row count)
    f = np.random.default_rng(n).standard_normal(shape)
    spacing = [1e-4, 1.1e-4]
    got = _abi.spectral_apply(f, spacing, 1, axis=along, kap=0.15 * spacing[0])
    want = _ref(f, spacing, 1, along, 0.15 * spacing[0], True, 0.0)
    assert _rel(got, want) < 2e-6 + 1.2e-7 * np.sqrt(LENGTHS[n]), _rel(got, want)


@pytest.mark.parametrize("shape", [(3001, 6), (6, 3001), (5, 2926), (33, 6), (6, 33)])
@pytest.mark.parametrize("absorb", [None, (0.5, 1.3)])
def test_routes_by_line_length_match_the_oracle(shape, absorb):
    """Lines whose jobs or axes do not fit LDS together (unfused updates, one job at a time)
    and lines that do: velocity and multi-row pressure sources, all records."""
    from kwave_amd.data import Vector
    from kwave_amd.kgrid import kWaveGrid
    from kwave_amd.kmedium import kWaveMedium
    from kwave_amd.ksensor import kSensor
    from kwave_amd.ksource import kSource
    from kwave_amd.solvers.kspace_solver import Simulation
    from oracle.kspace_ref import OracleSimulation

    rng = np.random.default_rng(3)
    dx = 1e-4
    kg = kWaveGrid(Vector(list(shape)), Vector([dx, dx]))
    kg.setTime(14, 0.3 * dx / 1700.0)
    med = kWaveMedium(sound_speed=1500.0 + 200.0 * rng.random(shape), density=1000.0 + 50.0 * rng.random(shape), BonA=6.0)
    if absorb:
        med.alpha_coeff, med.alpha_power = absorb
    src = kSource()
    mask = np.zeros(shape, dtype=bool)
    mask[shape[0] // 2, :: max(1, shape[1] // 5)] = True
    src.p_mask = src.u_mask = mask
    n = int(mask.sum())
    src.p = 1e4 * np.sin(0.4 * np.arange(9)[None, :] + 0.1 * np.arange(n)[:, None])
    src.uy = 0.02 * np.cos(0.3 * np.arange(7)[None, :] + 0.2 * np.arange(n)[:, None])
    sm = np.zeros(shape, dtype=bool)
    sm[::max(1, shape[0] // 9), :: max(1, shape[1] // 9)] = True
    sm |= mask
    sen = kSensor(sm)
    sen.record = ["p", "u", "p_final"]
    kw = dict(pml_size=(2, 2), pml_alpha=(2.0, 2.0))
    got = Simulation(kg, med, copy.deepcopy(src), sen, **kw).run()
    want = OracleSimulation(kg, med, copy.deepcopy(src), sen, **kw).run()
    for k in want:
        assert _rel(got[k], want[k]) < 1e-4, (k, _rel(got[k], want[k]))
