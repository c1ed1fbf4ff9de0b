"""What the first step measures for the segment height (SFV_TUNE_REPORT=1 prints
each measurement): nothing where the workgroup kernels run."""
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
