"""State downloads through the pinned staging slots (sfv_transfer.hip): states
just below and above the staged size, whole numbers of slots and one element
more, more chunks than slots, several threads at once (more than there are
lanes), and again after every handle was destroyed.  Bytes must come back
exactly."""
import threading

import numpy as np
import pytest

import volumefluxes as VF

from helpers import terrain

pytestmark = pytest.mark.gpu

MB = 1 << 20


def _sim(nx, ny, realtype=np.float64):
    sc = terrain(nx, ny, seed=1, realtype=realtype)
    return VF.Simulator(VF.HIPBackend(realtype), sc.system, sc.stepper, sc.grid, cfl=sc.cfl)


def _fill(sim, seed):
    U = sim.get_full_state()
    U = np.asfortranarray(np.random.default_rng(seed).standard_normal(U.shape).astype(U.dtype))
    sim.set_full_state(U)
    return U


# nx, ny with 4 ghost rows and columns: bytes = 3 * 8 * (nx + 4) * (ny + 4)
@pytest.mark.parametrize("nx,ny", [(508, 508), (587, 587), (588, 587), (1020, 1020), (1021, 1020), (509, 1363),
                                   (1277, 1399)])
def test_bytes(nx, ny):
    sim = _sim(nx, ny)
    U = _fill(sim, nx)
    print(f"[transfer] {nx}x{ny}: {U.nbytes / MB:.3f} MB", flush=True)
    for _ in range(2):
        assert np.array_equal(sim.get_full_state(), U)


def test_float32_and_interior():
    sim = _sim(1023, 701, np.float32)
    U = _fill(sim, 5)
    assert np.array_equal(sim.get_full_state(), U)
    h = VF.current_interior_state(sim)
    assert np.array_equal(np.asarray(h.h), U[2:-2, 2:-2, 0]) and np.array_equal(np.asarray(h.hu), U[2:-2, 2:-2, 1])


def test_threads():
    sims = [_sim(700 + 40 * k, 500) for k in range(7)]
    states = [_fill(s, k) for k, s in enumerate(sims)]
    bad = []

    def fetch(k):
        for _ in range(4):
            if not np.array_equal(sims[k].get_full_state(), states[k]):
                bad.append(k)

    threads = [threading.Thread(target=fetch, args=(k,)) for k in range(len(sims))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    del sims
    sim = _sim(700, 700)
    U = _fill(sim, 9)
    assert np.array_equal(sim.get_full_state(), U)
