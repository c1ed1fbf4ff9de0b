"""sfv_device_bytes_for against what handles hold: on the CPU the number of
state-sized buffers of each kind of run, on the GPU the bytes of a handle that
has run."""
import ctypes

import numpy as np
import pytest

import volumefluxes as VF
from volumefluxes import _capi as C

from helpers import make_hip, terrain

FE, RK = VF.ForwardEulerStepper(), VF.RungeKutta2()
NONE = VF.NoReconstruction()


def _bytes_for(cfg):
    return C.lib().sfv_device_bytes_for(ctypes.byref(cfg))


# state-sized buffers: three, and a fourth for ForwardEuler loops of one launch
# a step and for RungeKutta2 without the fused kernels
@pytest.mark.parametrize("stepper,bc,gc,nx,states", [
    (FE, VF.WallBC(), 2, 40, 4), (FE, VF.PeriodicBC(), 3, 40, 4), (FE, VF.NeumannBC(), 2, 40, 4),
    (FE, VF.NeumannBC(), 3, 40, 3), (FE, VF.WallBC(), 2, 1, 3), (FE, VF.WallBC(), 1, 40, 3),
    (RK, VF.WallBC(), 2, 40, 3), (RK, VF.NeumannBC(), 2, 40, 4), (RK, VF.WallBC(), 2, 1, 4), (RK, VF.WallBC(), 1, 40, 4)])
def test_states(stepper, bc, gc, nx, states):
    cfg = terrain(nx, 30, seed=1, stepper=stepper, bc=bc, gc=gc, rec=NONE if gc == 1 else None).config()
    nxT, nyT = nx + 2 * gc, 30 + 2 * gc
    want = states * 3 * nxT * nyT * 8 + (nxT + 1) * (nyT + 1) * 8
    assert want <= _bytes_for(cfg) <= want + 4096


def test_configurations_that_cannot_be_made():
    cfg = terrain(20, 30, seed=1, stepper=FE).config()
    for gc in (0, 9, 1000):
        cfg.gc = gc
        assert _bytes_for(cfg) > 0


@pytest.mark.gpu
@pytest.mark.parametrize("realtype", [np.float64, np.float32])
@pytest.mark.parametrize("bc", [VF.WallBC(), VF.PeriodicBC(), VF.NeumannBC()])
@pytest.mark.parametrize("stepper", [FE, RK])
@pytest.mark.parametrize("rain", [None, "table"])
def test_handles(stepper, bc, realtype, rain):
    sc = terrain(61, 33, seed=2, stepper=stepper, bc=bc, realtype=realtype)
    if rain:                                      # a table longer than a kilobyte, and a Horton factor
        sc.system.source_terms[1:] = [VF.TimeDependentRain(np.linspace(1.0, 9.0, 300), np.arange(300.0)),
                                      VF.HortonInfiltration(sc.grid, factor=np.ones(sc.grid.totalcells))]
    sim = make_hip(sc)
    VF.advance_steps(sim, 3)
    held, said = C.lib().sfv_device_bytes(sim.handle), _bytes_for(sim._cfg)
    print(f"[bytes] {type(stepper).__name__} {type(bc).__name__} {held} {said}", flush=True)
    assert held <= said <= held + 4096
