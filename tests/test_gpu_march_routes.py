"""The wave-march kernels where small grids would take the workgroup kernels:
the adjoint's forward and recomputed steps (stages 1, 2 and 4) on handles with
a set variant or segment height, and on a grid too large for workgroups; the
no-allocation call on such a grid.  Both families run the same arithmetic, so
the tolerance is zero."""
import ctypes

import numpy as np
import pytest

import volumefluxes as VF
from volumefluxes import _capi as C

from helpers import make_hip, terrain
from test_gpu_adjoint import _target
from test_oracle_ad import smooth_flow
from test_zz_no_alloc import DeviceArray, _hip

pytestmark = pytest.mark.gpu


def _gradient(sc, steps, every, kernels=None, rows=0):
    print(f"[adjoint] {sc.name} {kernels} rows={rows}", flush=True)
    sim = make_hip(sc, kernels)
    if rows:
        sim.set_march_rows(rows)
    r = VF.adjoint_gradient(sim, steps, _target(sc), checkpoint_every=every)
    return [np.asarray(r[k]) for k in ("J", "dJ_dB", "dJ_dCz", "dJ_dU0")] + [sim.get_full_state()]


def _same(a, b):
    assert all(np.array_equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("keep", [True, False])
@pytest.mark.parametrize("case", [dict(), dict(bc=VF.PeriodicBC(), dx=1.7), dict(gc=3, friction=False)])
def test_adjoint_with_a_set_variant(case, keep, monkeypatch):
    if not keep:                                  # every reverse step recomputes its own
        monkeypatch.setenv("SFV_ADJOINT_KEEP", "0")
    sc = smooth_flow(terrain(123, 46, seed=17, **case))
    want = _gradient(sc, 9, 4)
    for kernels, rows in [("march", 0), ("march", 3), ("tiled", 0), (None, 1), (None, 7), (None, 60)]:
        _same(_gradient(sc, 9, 4, kernels, rows), want)


def test_adjoint_of_a_larger_grid():
    sc = smooth_flow(terrain(661, 640, seed=18))
    _same(_gradient(sc, 5, 2), _gradient(sc, 5, 2, "tiled"))


@pytest.mark.parametrize("realtype,bc", [(np.float64, VF.WallBC()), (np.float32, VF.PeriodicBC())])
def test_noalloc_of_a_larger_grid(realtype, bc):
    hip = _hip()
    sc = terrain(661, 640, seed=19, realtype=realtype, bc=bc)
    sim = make_hip(sc, "per-pass")
    U0 = sim.get_full_state()
    VF.advance_steps(sim, 5)
    cfg = sc.config()
    B, U = DeviceArray(hip, sc.corners()), DeviceArray(hip, U0)
    print(f"[noalloc] {sc.name} {U0.dtype}", flush=True)
    try:
        t, dt = ctypes.c_double(0.0), ctypes.c_double(-1.0)
        assert C.lib().sfv_advance_noalloc(ctypes.byref(cfg), B.ptr, U.ptr, 5, float("inf"), ctypes.byref(t),
                                           ctypes.byref(dt), None) == C.SFV_OK, C.lib().sfv_create_error()
        got = U.get()
    finally:
        U.free()
        B.free()
    assert t.value == sim.t and dt.value == sim.current_timestep
    assert np.array_equal(got, sim.get_full_state())
