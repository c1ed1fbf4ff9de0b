"""Loops to an end time, queued a bounded number of steps ahead of what the
device reports, against the oracle: runs shorter and longer than that, step
limits below, at and above the run's length, a run that is over before it
starts, and single steps, whose time and dt come with their report.  The
arithmetic is the oracle's, so the tolerance is zero."""
import ctypes

import numpy as np
import pytest

import volumefluxes as VF
from volumefluxes import _capi as C

from helpers import make_hip, make_oracle, terrain

pytestmark = pytest.mark.gpu

CASES = {"rk2": {}, "euler": dict(stepper=VF.ForwardEulerStepper()), "neumann": dict(bc=VF.NeumannBC()),
         "euler_neumann": dict(stepper=VF.ForwardEulerStepper(), bc=VF.NeumannBC()), "f32": dict(realtype=np.float32),
         "gc1": dict(gc=1, rec=VF.NoReconstruction())}


def _run(sim, end, max_steps=0):
    t, n = ctypes.c_double(sim.t), ctypes.c_int64()
    C.check(sim.handle, C.lib().sfv_run(sim.handle, float(end), 1, 0.0, max_steps, ctypes.byref(t), ctypes.byref(n)))
    sim.t = t.value
    return n.value


@pytest.mark.parametrize("case", list(CASES))
def test_lengths(case):
    sc = terrain(70, 50, seed=12, **CASES[case])
    for k in (1, 2, 11, 12, 13, 25, 60):
        print(f"[loop] {case} {k}", flush=True)
        o, sim = make_oracle(sc), make_hip(sc)
        o.advance(k)
        end = o.t                                 # a run to this time takes k steps, the last one cut to it
        o = make_oracle(sc)
        assert _run(sim, end) == o.simulate_to_time(end)
        assert sim.t == end and np.array_equal(sim.get_full_state(), o.state())
        assert _run(sim, end) == 0                # over before it starts
        assert sim.t == end and np.array_equal(sim.get_full_state(), o.state())


@pytest.mark.parametrize("case", ["rk2", "euler", "euler_neumann"])
@pytest.mark.parametrize("limit", [1, 12, 13, 29, 30, 31])
def test_step_limits(case, limit):
    sc = terrain(70, 50, seed=13, **CASES[case])
    o, sim = make_oracle(sc), make_hip(sc)
    o.advance(30)
    end = o.t
    o = make_oracle(sc)
    assert _run(sim, end, limit) == o.simulate_to_time(end, max_steps=limit)
    assert sim.t == o.t and np.array_equal(sim.get_full_state(), o.state())


@pytest.mark.parametrize("case", list(CASES))
def test_single_steps(case):
    sc = terrain(64, 48, seed=14, **CASES[case])
    o, sim = make_oracle(sc), make_hip(sc)
    t = 0.0
    for k in range(9):
        limit = float("inf") if k % 2 else 1e-3
        dr = o.step(limit, t)
        assert VF.perform_step(sim, limit) == dr, k
        t = float(sc.realtype(sc.realtype(t) + sc.realtype(dr)))
        sim.t = t
        if k % 3 == 0:                            # otherwise the next step follows at once
            assert np.array_equal(sim.get_full_state(), o.state()), k
    assert np.array_equal(sim.get_full_state(), o.state())
