"""Relaxation of a field on itself (rel and bb one field).  Out of place, the sweeps
write the field every second time, and read their right-hand side from it as it then
is; a drop-in solver on one bound array takes each sweep's result as the next one's
right-hand side, as the oracle does on one array.  Tolerance: none."""
import ctypes

import numpy as np
import pytest

import impact_hip as ih
import oracle_lib as O

pytestmark = pytest.mark.gpu

W6, PYZ = (1,) * 6, (1, 1, -1, -1, -1, -1)
GRIDS = pytest.mark.parametrize("N,bc", [((33, 17, 17), W6), ((70, 11, 40), PYZ)])


def setup(N, bc):
    oc, gc = O.OracleCase(N, bc, (2.0, 1.0, 1.0), (0.0, 0.0, 0.0)), ih.Case(N, bc, (2.0, 1.0, 1.0))
    s = tuple(slice(oc.Sp[d] + 3, oc.Np[d] + 4) for d in (2, 1, 0))
    return oc, gc, s, np.random.default_rng(14).standard_normal(oc.shape)


@pytest.mark.parametrize("sweeps", [1, 2, 3, 4, 7])
@GRIDS
def test_jor(N, bc, sweeps):
    oc, gc, s, r = setup(N, bc)
    gc.upload(ih.PRE, r)
    gc.jor(sweeps, 0.8, oc.Sp, oc.Np, rel=ih.PRE, bb=ih.PRE)
    field, cur = r.copy(), r.copy()
    for n in range(sweeps):
        oc.jor(1, 0.8, oc.Sp, oc.Np, cur, field.copy(), oc.zeros())
        if n % 2:  # back in the field
            field = cur.copy()
    got = gc.download(ih.PRE)[s]
    assert np.array_equal(got, cur[s]), f"{int((got != cur[s]).sum())} values differ"
    gc.close()


@GRIDS
def test_drop_in_solver_on_one_bound_array(N, bc):
    oc, gc, s, r = setup(N, bc)
    want = r.copy()
    rc, sweeps = O.device_jacobi_solver(oc, 0.8, oc.Sp, oc.Np, want, want)
    mem = np.ascontiguousarray(r)
    ih.check(gc.lib.ih_bind_field(gc.h, ctypes.c_int(ih.PRE), ih._dp(mem)), "bind")
    assert gc.device_jacobi_solver(0.8, oc.Sp, oc.Np, mem, mem) == rc
    got = gc.download(ih.PRE)[s]
    assert np.array_equal(got, want[s]), f"{sweeps} sweeps, {int((got != want[s]).sum())} values differ"
    gc.close()
