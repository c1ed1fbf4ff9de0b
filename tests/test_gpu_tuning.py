"""What the first step measures for the segment height (SFV_TUNE_REPORT=1 prints
each measurement): nothing where the workgroup kernels run, else the kernels
that the steps take."""
import pytest

import volumefluxes as VF

from helpers import make_hip, terrain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernels,stepper,bc", [("hybrid", VF.RungeKutta2(), VF.WallBC()), (None, VF.RungeKutta2(), VF.WallBC()),
                                                ("hybrid", VF.ForwardEulerStepper(), VF.PeriodicBC()),
                                                (None, VF.ForwardEulerStepper(), VF.NeumannBC())])
def test_small_grids_measure_nothing(kernels, stepper, bc, monkeypatch, capfd):
    monkeypatch.setenv("SFV_TUNE_REPORT", "1")
    sim = make_hip(terrain(211, 173, seed=3, stepper=stepper, bc=bc), kernels)
    VF.advance_steps(sim, 2)
    assert "[sfv autotune]" not in capfd.readouterr().err
    assert sim.march_rows > 0


def _measured(capfd):
    return [line.split(", ")[1].split(":")[0] for line in capfd.readouterr().err.splitlines() if "[sfv autotune]" in line]


# sizes that no other test takes (heights are kept per size class)
@pytest.mark.parametrize("nx,ny,stepper,bc,first,then", [
    (5000, 110, VF.ForwardEulerStepper(), VF.WallBC(), ["stage 1"], ["stage 3"]),
    (5000, 131, VF.ForwardEulerStepper(), VF.NeumannBC(), ["stage 1"], ["stage 3"]),
    (5000, 156, VF.RungeKutta2(), VF.NeumannBC(), ["stage 1"], []),
    (5000, 186, VF.RungeKutta2(), VF.WallBC(), ["steps"], [])])
def test_the_kernels_that_run(nx, ny, stepper, bc, first, then, monkeypatch, capfd):
    monkeypatch.setenv("SFV_TUNE_REPORT", "1")
    sim = make_hip(terrain(nx, ny, seed=4, stepper=stepper, bc=bc))
    VF.perform_step(sim, float("inf"))
    assert _measured(capfd) == first
    for _ in range(2):
        VF.advance_steps(sim, 3)
        assert _measured(capfd) == then
        then = []
    sim2 = make_hip(terrain(nx, ny, seed=4, stepper=stepper, bc=bc))
    VF.advance_steps(sim2, 3)                     # kept for the size class
    assert _measured(capfd) == [] and sim2.march_rows == sim.march_rows
    sim2.set_march_rows(5)
    VF.perform_step(sim2, float("inf"))
    VF.advance_steps(sim2, 3)
    assert _measured(capfd) == [] and sim2.march_rows == 5
