"""The small-grid forms of the step kernels give the bits of the large-grid ones.

A size rule switches between the two (kw_col_pass.hip), so a batch and its instances
run alone, or a step before and after its sources end, may run different forms.
"""
import copy

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _case(shape, absorb, bona):
    """Multi-row pressure and velocity sources, heterogeneous medium, every record."""
    from kwave_amd.data import Vector
    from kwave_amd.kgrid import kWaveGrid
    from kwave_amd.kmedium import kWaveMedium
    from kwave_amd.ksensor import kSensor
    from kwave_amd.ksource import kSource

    rng = np.random.default_rng(11)
    dx = 1e-4
    kg = kWaveGrid(Vector(list(shape)), Vector([dx] * len(shape)))
    kg.setTime(24, 0.3 * dx / 1700.0)
    med = kWaveMedium(sound_speed=1500.0 + 200.0 * rng.random(shape), density=1000.0 + 50.0 * rng.random(shape))
    if absorb:
        med.alpha_coeff, med.alpha_power = absorb
    if bona:
        med.BonA = bona
    src = kSource()
    sl = tuple(slice(n // 2 - 2, n // 2 + 2) for n in shape)
    pm = np.zeros(shape, dtype=bool)
    pm[sl] = True
    src.p_mask = src.u_mask = pm
    n = int(pm.sum())
    src.p = 1e4 * np.sin(0.4 * np.arange(12)[None, :] + 0.1 * np.arange(n)[:, None])
    src.ux = 0.05 * np.cos(0.3 * np.arange(9)[None, :])
    sm = np.zeros(shape, dtype=bool)
    sm[tuple(slice(n // 4, 3 * n // 4) for n in shape[:-1]) + (slice(None, None, 3),)] = True
    sen = kSensor(sm)
    sen.record = ["p", "u_staggered", "p_final", "u_final"]
    return kg, med, src, sen


@pytest.mark.parametrize("shape,absorb,bona", [
    ((16, 24), None, None),              # the shortest lines of each family
    ((128, 128), None, None),
    ((128, 40), (0.5, 1.3), 6.0),
    ((512, 56), (0.02, 2.0), None),      # two wavefronts per tile
    ((640, 16), (0.5, 1.5), None),
    ((1024, 32), (0.5, 1.1), 6.0),       # the longest lines, four wavefronts per tile
    ((24, 32, 40), (0.5, 1.3), 6.0),
    ((48, 112, 16), None, 6.0),
    ((32, 16, 768), (0.5, 1.5), None),
])
def test_small_grid_forms_give_the_same_bits(shape, absorb, bona, monkeypatch):
    from kwave_amd.solvers.kspace_solver import Simulation

    kg, med, src, sen = _case(shape, absorb, bona)

    def run(small):
        monkeypatch.setenv("KW_COL_SMALL", small)
        monkeypatch.setenv("KW_Z_SMALL", small)
        return Simulation(kg, med, copy.deepcopy(src), sen, pml_size=(3,) * len(shape), pml_alpha=(2.0,) * len(shape)).run()

    large = run("0")
    assert all(np.abs(v).max() > 0 for v in large.values())
    for form in ("1", "2"):
        for k, v in run(form).items():
            assert np.array_equal(v, large[k]), (form, k)


@pytest.mark.parametrize("shape", [(70, 66), (128, 64), (20, 18, 16), (32, 16, 24)])
@pytest.mark.parametrize("sensor", ["all", "few"])
def test_records_do_not_depend_on_how_steps_are_grouped(shape, sensor, monkeypatch):
    """Steps run in captured blocks gather a step's sensors in the next step's first column
    pass; run(), step() and the graph-free path record the same bits, with few sensors (one
    workgroup gathers and advances the counter) and with more than 4096 (two launches)."""
    from kwave_amd.solvers.kspace_solver import Simulation

    kg, med, src, sen = _case(shape, (0.5, 1.3), None)
    if sensor == "all":
        sen.mask = np.ones(shape, dtype=bool)
    sen.record = ["p", "p_max", "u", "u_staggered", "p_final"]
    sen.record_start_index = 3

    def make():
        return Simulation(kg, med, copy.deepcopy(src), sen, pml_size=(3,) * len(shape), pml_alpha=(2.0,) * len(shape))

    blocks = make().run()
    sim = make()
    sim.setup()
    while sim.t < sim.Nt:
        sim.step()
    monkeypatch.setenv("KW_NO_GRAPH", "1")
    for other in (sim.run(), make().run()):
        for k, v in blocks.items():
            assert np.array_equal(v, other[k]), k


@pytest.mark.parametrize("shape,absorb,bona,mode", [
    ((16, 24), None, None, "additive"),
    ((70, 128), (0.5, 1.3), 6.0, "dirichlet"),
    ((128, 56), (0.02, 2.0), 6.0, "additive"),  # Stokes
    ((32, 1024), (0.5, 1.1), None, "additive"),  # two wavefronts per row pair
    ((24, 32, 40), (0.5, 1.3), 6.0, "additive"),
    ((16, 14, 64), None, 6.0, "dirichlet"),
])
def test_small_grid_forms_of_the_reverse_sweep_give_the_same_bits(shape, absorb, bona, mode, monkeypatch):
    from kwave_amd.adjoint import sound_speed_gradient

    kg, med, src, sen = _case(shape, absorb, bona)
    src.p_mode = mode
    sen.record = ["p"]
    adj = np.random.default_rng(3).standard_normal((int(sen.mask.sum()), 24)).astype(np.float32)

    def run(small):
        monkeypatch.setenv("KW_Z_SMALL", small)
        return sound_speed_gradient(kg, med, copy.deepcopy(src), sen, adj, pml_size=(3,) * len(shape),
                                    pml_alpha=(2.0,) * len(shape), checkpoint=7)[0]

    large = run("0")
    assert np.abs(large).max() > 0
    assert np.array_equal(run("2"), large)


@pytest.mark.parametrize("shape", [(64, 512, 512), (16, 1024, 1024), (96, 448, 384), (160, 320, 320)])
def test_the_momentum_order_of_large_grids_gives_the_same_bits(shape, monkeypatch):
    """Above 14 million elements the tables are staged before the loads."""
    from kwave_amd import _abi
    from kwave_amd.solvers.plan import DevicePlan
    from kwave_amd.solvers.setup import build_instance

    kg, med, src, sen = _case(shape, None, None)
    sm = np.zeros(shape, dtype=bool)
    sm[tuple(slice(n // 2 - 4, n // 2 + 4) for n in shape)] = True
    sen.mask, sen.record = sm, ["p", "u_staggered"]
    st = build_instance(kg, med, src, sen, pml_size=(3,) * 3, pml_alpha=(2.0,) * 3)

    def run(small):
        monkeypatch.setenv("KW_Z_SMALL", small)
        pl = DevicePlan([st])
        pl.run(4)
        out = [pl.field(0, f) for f in (_abi.F_P, _abi.F_UX, _abi.F_UX + 1, _abi.F_UX + 2)]
        pl.close()
        return out

    for a, b in zip(run("1"), run("2")):  # "2": the small-grid form at any size
        assert np.abs(a).max() > 0 and np.array_equal(a, b)


@pytest.mark.parametrize("shape", [(24, 16, 56), (16, 24, 112), (16, 16, 224), (24, 16, 448), (16, 16, 1024)])
@pytest.mark.parametrize("absorb,bona", [(None, None), ((0.02, 2.0), 6.0), ((0.5, 1.3), 6.0)])
def test_small_grid_forms_of_the_longest_rows_in_3d(shape, absorb, bona, monkeypatch):
    """Three groups of lanes where their exchanges take the most LDS (fourteen elements a lane)
    and, at 1024, two wavefronts a group: the step's forms and the reverse sweep's."""
    from kwave_amd.adjoint import sound_speed_gradient
    from kwave_amd.solvers.kspace_solver import Simulation

    kg, med, src, sen = _case(shape, absorb, bona)
    pml = dict(pml_size=(3,) * 3, pml_alpha=(2.0,) * 3)
    adj = np.random.default_rng(3).standard_normal((int(sen.mask.sum()), 24)).astype(np.float32)

    def run(form):
        monkeypatch.setenv("KW_COL_SMALL", form)
        monkeypatch.setenv("KW_Z_SMALL", form)
        out = Simulation(kg, med, copy.deepcopy(src), sen, **pml).run()
        sen_p = copy.deepcopy(sen)
        sen_p.record = ["p"]
        out["gradient"] = sound_speed_gradient(kg, med, copy.deepcopy(src), sen_p, adj, checkpoint=7, **pml)[0]
        return out

    large = run("0")
    for k, v in run("2").items():
        assert np.abs(large[k]).max() > 0 and np.array_equal(v, large[k]), k
