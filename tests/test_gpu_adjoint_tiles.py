"""The adjoint's face kernel (workgroups of 63 columns by 4 rows of faces) and
its recomputed steps (three launches, one prepared loop per segment) at the
edges of their tiles and segments, against the oracle's forward-mode
derivative as in test_gpu_adjoint.py.  Both are exact derivatives of the same
branches: they agree to rounding, 1e-9 over a few smooth steps."""
import numpy as np
import pytest

import volumefluxes as VF
from volumefluxes.scenarios import terrain_initial_state, terrain_topography

from helpers import Scenario, _system, terrain
from test_gpu_adjoint import _check
from test_oracle_ad import smooth_flow

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(61, 3), (62, 4), (63, 5), (125, 7), (126, 8), (127, 9)])
@pytest.mark.parametrize("bc", [VF.WallBC(), VF.PeriodicBC()])
def test_tile_edges(nx, ny, bc):
    print(f"[adjoint] {nx}x{ny} {type(bc).__name__}", flush=True)
    _check(smooth_flow(terrain(nx, ny, seed=nx + ny, bc=bc, n_bumps=6)), 5, 2, dirs=1)


# steps and checkpoint spacings: one segment, a last segment of one step, odd
# segment starts (the kept steps take the other slot)
@pytest.mark.parametrize("steps,every", [(1, 1), (4, 9), (7, 3), (10, 5), (9, 1)])
def test_segments(steps, every):
    _check(smooth_flow(terrain(70, 33, seed=31)), steps, every, dirs=1)


@pytest.mark.parametrize("gc,dx", [(3, 1.7), (4, 0.5), (2, 2.5)])
def test_ghosts_and_spacings(gc, dx):
    _check(smooth_flow(terrain(66, 30, seed=37, gc=gc, dx=dx)), 6, 4, dirs=2)


def test_rain_changes_between_steps():
    """A recomputed step's second stage takes the rain of its own start."""
    nx, ny = 64, 40
    grid = VF.CartesianGrid(nx, ny, gc=2, boundary=VF.WallBC(), extent=[[0.0, 1.0 * nx], [0.0, 1.0 * ny]])
    B = terrain_topography(grid, seed=9, n_bumps=8, amp=(0.5, 2.0), width=(6.0, 20.0))
    rain = VF.TimeDependentRain([36.0, 0.0, 90.0, 5.0], [0.0, 0.02, 0.05, 0.13])
    system = _system(grid, B, sources=[VF.SourceTermBottom(), rain], friction=VF.ImplicitFriction(Cz=0.03 * 0.03),
                     kappa=1e-4)
    sc = Scenario("rain_table", grid, system, VF.RungeKutta2(), 0.25, terrain_initial_state(grid, B, 4.0), np.float64, B)
    _check(smooth_flow(sc), 12, 5, dirs=1)
