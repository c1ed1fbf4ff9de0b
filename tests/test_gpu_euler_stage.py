"""The ForwardEuler stage (one launch finishes a step and finds the next one's
right-hand side) against the oracle, bit for bit: each boundary condition,
workgroup and wave-march kernels, the specialised and general instantiations,
one, two and three steps (the loop's first and last step take other launches),
and loops that end by time, by step count and by both.  Every arithmetic step
is the oracle's, so the tolerance is zero; only Horton's exp may differ in its
last bit, and is compared with the per-pass kernels, which call the same exp."""
import numpy as np
import pytest

import volumefluxes as VF

from helpers import Scenario, _system, make_hip, make_oracle, terrain
from volumefluxes.scenarios import terrain_initial_state, terrain_topography

pytestmark = pytest.mark.gpu

FE = VF.ForwardEulerStepper()


def _advance_both(sc, steps, kernels=None):
    print(f"[euler] {sc.name} steps={steps}", flush=True)
    o, sim = make_oracle(sc), make_hip(sc, kernels)
    for n in steps:                     # the state, ghosts and corners included, after each loop
        o.advance(n)
        VF.advance_steps(sim, n)
        assert sim.t == o.t, n
        assert np.array_equal(sim.get_full_state(), o.state()), n
    return sim


@pytest.mark.parametrize("bc", [VF.WallBC(), VF.PeriodicBC(), VF.NeumannBC()])
@pytest.mark.parametrize("nx,ny", [(40, 37), (60, 1 + 60), (121, 75), (700, 620), (900, 610)])
def test_steps(nx, ny, bc):
    sim = _advance_both(terrain(nx, ny, seed=nx + ny, bc=bc, stepper=FE), (1, 2, 3, 4) if nx < 500 else (1, 3))
    assert sim.kernels == "hybrid"


@pytest.mark.parametrize("case", ["f32", "neumann_f32", "gc3", "neumann_gc3", "periodic_gc4", "dx1.7", "dx0.3_f32",
                                  "no_friction", "norec", "narrow"])
def test_instantiations(case):
    kw = dict(seed=len(case), stepper=FE)
    shape = (97, 66)
    if "f32" in case:
        kw["realtype"] = np.float32
    if "neumann" in case:
        kw["bc"] = VF.NeumannBC()
    if "gc3" in case:
        kw["gc"] = 3
    if "gc4" in case:
        kw.update(gc=4, bc=VF.PeriodicBC())
    if "dx" in case:
        kw["dx"] = float(case.split("_")[0][2:])
    if case == "no_friction":
        kw["friction"] = False
    if case == "norec":
        kw["rec"] = VF.NoReconstruction()
    if case == "narrow":                # ghosts whose sources are ghosts: the three-launch step
        shape = (1, 66)
    _advance_both(terrain(*shape, **kw), (3, 8))


@pytest.mark.parametrize("rows", [1, 3, 40])
def test_forced_heights(rows):
    sc = terrain(150, 47, seed=3, bc=VF.NeumannBC(), stepper=FE)
    o, sim = make_oracle(sc), make_hip(sc)
    sim.set_march_rows(rows)
    o.advance(5)
    VF.advance_steps(sim, 5)
    assert np.array_equal(sim.get_full_state(), o.state())


@pytest.mark.parametrize("bc", [VF.PeriodicBC(), VF.NeumannBC()])
def test_loops_ending_by_time(bc):
    sc = terrain(90, 50, seed=8, bc=bc, stepper=FE)
    o, sim = make_oracle(sc), make_hip(sc)
    for t in (0.05, 0.06, 0.9):
        o.simulate_to_time(t)
        VF.simulate_to_time(sim, t)
        assert sim.t == o.t == t
        assert np.array_equal(sim.get_full_state(), o.state()), t


@pytest.mark.parametrize("bc", [VF.WallBC(), VF.NeumannBC()])
@pytest.mark.parametrize("realtype", [np.float64, np.float32])
def test_horton_and_rain_table(bc, realtype):
    """Rates that change with time: the stage finds the next step's rates itself.
    (The end time is a float32 value: a Float32 run stops short of any other.)"""
    nx, ny = 107, 80
    grid = VF.CartesianGrid(nx, ny, gc=2, boundary=bc, extent=[[0.0, 1.0 * nx], [0.0, 1.0 * ny]])
    B = terrain_topography(grid, seed=5, n_bumps=16, amp=(0.5, 5.0), width=(4.0, 20.0))
    factor = np.abs(np.random.default_rng(3).standard_normal((nx + 4, ny + 4)))
    rain = VF.TimeDependentRain([36.0, 0.0, 90.0], [0.0, 0.2, 0.5])
    states = []
    for kernels in (None, "per-pass"):
        sys_ = _system(grid, B, sources=[VF.SourceTermBottom(), rain, VF.HortonInfiltration(grid, factor=factor)],
                       friction=VF.ImplicitFriction(Cz=0.03 * 0.03))
        sim = make_hip(Scenario("horton", grid, sys_, FE, 0.25, terrain_initial_state(grid, B, 2.0), realtype, B), kernels)
        VF.simulate_to_time(sim, 0.75)
        states.append((sim.t, sim.get_full_state()))
    assert states[0][0] == states[1][0]
    assert np.array_equal(states[0][1], states[1][1])
