"""State downloads of the staged size into memory that the runtime allocated:
pinned host memory and device memory (sfv_get_state's destination, as a plain
copy takes it).  Bytes must come back exactly."""
import ctypes

import numpy as np
import pytest

from volumefluxes import _capi as C

from test_gpu_transfer import _fill, _sim
from test_zz_no_alloc import D2H, _hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["pinned", "device"])
def test_known_destination(kind):
    sim = _sim(900, 700)
    U = _fill(sim, 3)
    hip = _hip()
    p = ctypes.c_void_p()
    if kind == "pinned":
        hip.hipHostMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t, ctypes.c_uint]
        assert hip.hipHostMalloc(ctypes.byref(p), U.nbytes, 0) == 0
    else:
        assert hip.hipMalloc(ctypes.byref(p), U.nbytes) == 0
    print(f"[transfer] {kind} destination, {U.nbytes} bytes", flush=True)
    try:
        C.check(sim.handle, C.lib().sfv_get_state(sim.handle, p, C.SFV_LAYOUT_FULL))
        out = np.empty_like(U, order="F")
        assert hip.hipMemcpy(out.ctypes.data_as(ctypes.c_void_p), p, U.nbytes, D2H if kind == "device" else 0) == 0
    finally:
        if kind == "pinned":
            hip.hipHostFree.argtypes = [ctypes.c_void_p]
            hip.hipHostFree(p)
        else:
            hip.hipFree(p)
    assert np.array_equal(out, U)
