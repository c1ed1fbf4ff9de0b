"""The workgroup kernels (one workgroup per strip segment, swe_kernels_block.hip)
against the oracle, bit for bit: grids whose segment heights take each
workgroup size (6, 10 and 16 waves, one and two chunks of rows), heights that
end inside a chunk, the specialised and general instantiations, and inputs
that make a workgroup leave the ranged forms in the middle of its segment.
Every arithmetic step is the oracle's, so the tolerance is zero."""
import numpy as np
import pytest

import volumefluxes as VF
from volumefluxes.scenarios import cell_bottom, terrain_initial_state, terrain_topography

from helpers import Scenario, _system, make_hip, make_oracle, run_both_compare, terrain

pytestmark = pytest.mark.gpu


def _check(sc, steps, kernels="tiled"):
    print(f"[block] {sc.name} {kernels}", flush=True)
    dts, U_hip, U_ref = run_both_compare(sc, steps, kernels=kernels)
    assert all(dh == dr for dh, dr in dts), sc.name
    assert np.array_equal(U_hip, U_ref), sc.name


# strips x heights: 1 row (6 waves), 2 rows of 4 strips, 6 (10 waves), 12 (16
# waves), 24 (two chunks of 16), a last segment of one row
@pytest.mark.parametrize("nx,ny", [(64, 48), (200, 130), (333, 221), (420, 421), (600, 600), (61, 259)])
def test_workgroup_heights(nx, ny):
    sc = terrain(nx, ny, seed=nx + ny)
    _check(sc, 4)
    sim = make_hip(sc)
    VF.perform_step(sim, float("inf"))
    assert sim.kernels == "tiled"                 # chosen without being asked for


def test_larger_grid_runs_in_several_rounds():
    _check(terrain(900, 700, seed=5), 2)


def _options(dx, rho, infiltration, bc, realtype, friction=True):
    nx, ny = 130, 75
    grid = VF.CartesianGrid(nx, ny, gc=2, boundary=bc, extent=[[0.0, nx * dx], [0.0, ny * dx]])
    B = terrain_topography(grid, seed=77, n_bumps=16, amp=(0.5, 5.0), width=(4.0 * dx, 20.0 * dx))
    eq = VF.ShallowWaterEquations(VF.BottomTopography2D(B, None, grid), rho=rho, desingularizing_kappa=1e-4)
    sources = [VF.SourceTermBottom(), VF.ConstantRain(0.036)]
    if infiltration:
        sources.insert(0, VF.ConstantInfiltration(2e-6))
    system = VF.ConservedSystem(None, VF.LinearReconstruction(), VF.CentralUpwind(eq), eq, grid, sources,
                                VF.ImplicitFriction(Cz=0.03 * 0.03) if friction else None)
    return Scenario(f"dx{dx}_rho{rho}_{infiltration}", grid, system, VF.RungeKutta2(), 0.25,
                    terrain_initial_state(grid, B, 2.0), realtype, B)


@pytest.mark.parametrize("kernels", ["tiled", "march"])
@pytest.mark.parametrize("case", [(1.0, 1.0, True, VF.WallBC(), np.float64), (1.7, 1.0, False, VF.PeriodicBC(), np.float64),
                                  (0.3, 1.0, True, VF.WallBC(), np.float32), (1.0, 2.5, False, VF.WallBC(), np.float64),
                                  (3.1, 1.0, True, VF.WallBC(), np.float64, False)])
def test_instantiations(case, kernels):
    """Power-of-two and other spacings, infiltration, no friction (the
    specialised kernels) and a density other than 1 (the general ones)."""
    _check(_options(*case), 15, kernels)


@pytest.mark.parametrize("value", [1e-40, -3e-35, 5e-324, 1e13])
def test_out_of_band_values_mid_segment(value):
    sc = terrain(150, 90, seed=41)
    depth = sc.U0[:, :, 0] - cell_bottom(sc.B)[2:-2, 2:-2]
    cells = np.argwhere(depth > 0.5)
    rng = np.random.default_rng(1)
    U0 = sc.U0.copy()
    for k, (i, j) in enumerate(cells[rng.choice(len(cells), 5, replace=False)]):
        U0[i, j, 1 + (k % 2)] = value
    sc.U0 = U0
    _check(sc, 3 if abs(value) > 1 else 12)


@pytest.mark.parametrize("kernels", ["tiled", "march"])
def test_momenta_near_the_friction_bound(kernels):
    """Momenta around 2^-80 and 2^-120, where the ranged friction and face
    forms give way to the general ones."""
    sc = terrain(96, 64, seed=43)
    U0 = sc.U0.copy()
    rng = np.random.default_rng(2)
    for e in (-78, -80, -82, -118, -120, -122):
        i, j = int(rng.integers(8, 88)), int(rng.integers(8, 56))
        U0[i, j, 1], U0[i, j, 2] = 1.3 * 2.0 ** e, -1.7 * 2.0 ** e
    sc.U0 = U0
    _check(sc, 8, kernels)
