"""An error of the runtime that the caller has not looked at yet: a transfer neither
reports it as its own nor clears it, from pinned and from other memory (the device
asked for does not exist, which the runtime refuses on the host)."""
import ctypes

import numpy as np
import pytest

import impact_hip as ih

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pinned", [False, True])
def test_transfers_leave_a_pending_error(pinned):
    c = ih.Case((33, 17, 17), (1,) * 6)
    hip, mem = c.lib, ctypes.c_void_p()
    if pinned:
        assert hip.hipHostMalloc(ctypes.byref(mem), ctypes.c_size_t(8 * int(np.prod(c.shape))), 0) == 0
        a = np.ctypeslib.as_array(ctypes.cast(mem, ctypes.POINTER(ctypes.c_double)), c.shape)
    else:
        a = np.empty(c.shape)
    a[...] = np.random.default_rng(21).standard_normal(c.shape)
    want = a.copy()
    hip.hipGetLastError()
    error = hip.hipSetDevice(9999)
    assert error != 0 and hip.hipPeekAtLastError() == error
    for first in (True, False):  # the first transfer allocates the buffer
        assert hip.ih_field_upload(c.h, ih.PRE, ih._dp(a)) == 0
        assert hip.hipPeekAtLastError() == error
        a[...] = 0.0
        assert hip.ih_field_download(c.h, ih.PRE, ih._dp(a)) == 0
        assert hip.hipGetLastError() == error
        assert np.array_equal(a, want)
        if first:
            assert hip.hipSetDevice(9999) == error
    assert hip.hipGetLastError() == 0
    if pinned:
        hip.hipHostFree(mem)
    c.close()
