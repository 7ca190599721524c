"""Host arrays of the calls that take them.  Transfers of a whole field from and to
memory that is not pinned, through one or several fills of the case's buffer and
beside pinned arrays; device_jacobi_solver, whose sweeps between two stopping
tests are one call over the whole range and a call each elsewhere, against the
oracle's.  Tolerance: none (copies; the oracle's operations in its order)."""
import ctypes

import numpy as np
import pytest

import impact_hip as ih
import oracle_lib as O

pytestmark = pytest.mark.gpu

W6 = (1, 1, 1, 1, 1, 1)


# 27 KB; the 4 MiB of the buffer; a fill and a remainder
@pytest.mark.parametrize("N", [(8, 8, 8), (57, 121, 57), (118, 71, 91), (505, 9, 129)])
@pytest.mark.parametrize("pinned", [False, True])
def test_whole_fields_round_trip(N, pinned):
    c = ih.Case(N, W6)
    mem = [ctypes.c_void_p(), ctypes.c_void_p()]
    if pinned:  # by the runtime that the library is linked with
        for m in mem:
            assert c.lib.hipHostMalloc(ctypes.byref(m), ctypes.c_size_t(8 * int(np.prod(c.shape))), 0) == 0
        a, out = (np.ctypeslib.as_array(ctypes.cast(m, ctypes.POINTER(ctypes.c_double)), c.shape) for m in mem)
    else:
        a, out = np.empty(c.shape), np.empty(c.shape)
    a[...] = np.random.default_rng(7).standard_normal(c.shape)
    c.upload(ih.PRE, a)
    for lo in ((-3, -3, -3), tuple(n + 3 for n in N)):  # the outermost ghost points
        one = c.get_box(ih.PRE, lo, lo)
        assert one.ravel()[0] == a[tuple(lo[d] + 3 for d in (2, 1, 0))]
    ih.check(c.lib.ih_field_download(c.h, ih.PRE, ih._dp(out)), "download")
    assert np.array_equal(out, a)
    for m in mem:
        if m:
            c.lib.hipHostFree(m)
    c.close()


@pytest.mark.parametrize("spec", [((33, 17, 17), W6, None), ((12, 11, 10), (1, 1, -1, -1, -1, -1), None),
                                  ((12, 10, 11), (-1, -1, 1, 1, 1, 1), None), ((17, 13, 11), W6, ((2, 2, 2), (16, 11, 10))),
                                  ((600, 9, 9), W6, None)],
                         ids=["walls", "periodic-yz", "periodic-x", "sub-box", "long-rows"])
def test_drop_in_solver(spec):
    N, bc, box = spec
    oc, gc = O.OracleCase(N, bc, (2.0, 1.0, 1.0), (0.0, 0.0, 0.0)), ih.Case(N, bc, (2.0, 1.0, 1.0))
    ss, nn = box or (oc.Sp, oc.Np)
    rng = np.random.default_rng(8)
    bb, want = rng.standard_normal(oc.shape), rng.standard_normal(oc.shape)
    got = want.copy()
    rc, sweeps = O.device_jacobi_solver(oc, 0.8, ss, nn, want, bb)
    gc.fill(ih.COMP, np.nan)  # what its scratch held before is not read
    assert gc.device_jacobi_solver(0.8, ss, nn, got, bb.copy()) == rc == 0
    s = tuple(slice(oc.Sp[d] + 3, oc.Np[d] + 4) for d in (2, 1, 0))
    assert np.array_equal(got[s], want[s]), f"{sweeps} sweeps"
    gc.close()
