"""Loops to an end time whose steps last longer than the host polls before it
asks the stream (200 us): the number of steps, the end and the state are those
of the same steps taken by count, the last one cut to the end time.  The
arithmetic is the same, so the tolerance is zero."""
import ctypes

import numpy as np
import pytest

import volumefluxes as VF
from volumefluxes import _capi as C

from helpers import make_hip, terrain
from test_gpu_run_loop import _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", ["rk2", "per-pass", "euler"])
@pytest.mark.parametrize("steps", [1, 12, 29])
def test_long_steps(case, steps):
    # the per-pass steps of 1500^2 and the ForwardEuler steps of 3000^2 last as long as RK2's of 2048^2
    n = {"rk2": 2048, "per-pass": 1500, "euler": 3000}[case]
    sc = terrain(n, n, seed=2, stepper=VF.ForwardEulerStepper() if case == "euler" else None)
    kernels = "per-pass" if case == "per-pass" else None
    print(f"[loop] {case} {n}^2, {steps} steps", flush=True)
    a, b = make_hip(sc, kernels), make_hip(sc, kernels)
    VF.advance_steps(a, steps - 1)
    dt = VF.perform_step(a, float("inf"))
    end = a.t + 0.5 * dt                          # in the middle of the last step
    a = make_hip(sc, kernels)
    VF.advance_steps(a, steps - 1)
    assert VF.perform_step(a, end - a.t) == end - a.t
    assert _run(b, end) == steps
    last = ctypes.c_double()
    C.check(b.handle, C.lib().sfv_current_timestep(b.handle, ctypes.byref(last)))
    assert b.t == a.t + a.current_timestep and last.value == a.current_timestep
    assert np.array_equal(a.get_full_state(), b.get_full_state())
    assert _run(b, end) == 0
