"""The memory that large downloads are staged through stays with a server: a
request of 8 MB or more makes it, requests without a large state that follow
do not take it away."""
import ctypes

import numpy as np
import pytest

import volumefluxes as VF
from volumefluxes import _capi as C

from helpers import terrain

pytestmark = pytest.mark.gpu


def _lanes():
    f = C.lib()["_ZN3sfv13staging_lanesEv"]       # sfv::staging_lanes(), no part of the C interface
    f.restype = ctypes.c_int
    return f()


def _serve(server, nx, ny):
    sc = terrain(nx, ny, seed=nx)
    print(f"[serving] {nx}x{ny}", flush=True)
    rid = server.submit(sc.system, sc.grid, sc.U0, 0.02)
    assert server.wait(rid, timeout=60)["status"] == C.SFV_REQ_DONE
    assert np.isfinite(server.fetch(rid)[0]).all()


def test_lane_stays_with_the_server():
    with VF.Server(4 << 30) as server:
        for nx, ny in [(700, 640), (64, 48), (80, 60), (700, 640), (50, 40)]:
            _serve(server, nx, ny)
            assert _lanes() >= 1, (nx, ny)
