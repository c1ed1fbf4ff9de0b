"""A state restored verbatim whose ghost cells are not what the boundary
condition gives: NeumannBC handles, and RungeKutta2 on the hybrid kernels,
take them as given in the next step, as the per-pass kernels do, and the
boundary condition's after it.  The arithmetic is the same, so the tolerance
is zero."""
import numpy as np
import pytest

import volumefluxes as VF

from helpers import make_hip, terrain

pytestmark = pytest.mark.gpu


def _restored(sc, kernels, rows, seed):
    sim = make_hip(sc, kernels)
    if rows:
        sim.set_march_rows(rows)
    U = sim.get_full_state()
    g = sc.grid.gc
    rng = np.random.default_rng(seed)
    ghost = np.ones(U.shape[:2], bool)
    ghost[g:-g, g:-g] = False
    U[ghost, 0] += rng.uniform(0.0, 1.0, ghost.sum()).astype(U.dtype)
    U[ghost, 1:] = rng.uniform(-0.5, 0.5, (ghost.sum(), 2)).astype(U.dtype)
    sim.set_full_state(U)
    return sim


def _compare(sc, kernels, rows):
    for go in (lambda s: VF.perform_step(s, float("inf")), lambda s: VF.advance_steps(s, 1),
               lambda s: VF.advance_steps(s, 4), lambda s: VF.simulate_to_time(s, 0.5)):
        a, b = _restored(sc, kernels, rows, 5), _restored(sc, "per-pass", 0, 5)
        for _ in range(2):
            go(a)
            go(b)
            assert a.t == b.t and a.current_timestep == b.current_timestep
            assert np.array_equal(a.get_full_state(), b.get_full_state())


@pytest.mark.parametrize("stepper", [VF.ForwardEulerStepper(), VF.RungeKutta2()])
@pytest.mark.parametrize("gc", [2, 3])
@pytest.mark.parametrize("realtype", [np.float64, np.float32])
@pytest.mark.parametrize("rows", [0, 5])              # workgroup and wave-march kernels
def test_neumann(stepper, gc, realtype, rows):
    _compare(terrain(131, 47, seed=gc, bc=VF.NeumannBC(), stepper=stepper, gc=gc, realtype=realtype), None, rows)


@pytest.mark.parametrize("bc", [VF.WallBC(), VF.PeriodicBC()])
@pytest.mark.parametrize("rows", [0, 5])
def test_hybrid(bc, rows):
    _compare(terrain(131, 47, seed=9, bc=bc), "hybrid", rows)
