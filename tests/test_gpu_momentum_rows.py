"""The single-term momentum calls, four planes a thread: every remainder of the
planes and of the 64-point rows, each component and direction, in place on NL as a
host calls them.  Tolerance: none (the oracle's operations in its order)."""
import numpy as np
import pytest

import impact_hip as ih
import oracle_lib as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n3", [8, 9, 10, 11, 13])
@pytest.mark.parametrize("n1,bc", [(64, (1,) * 6), (65, (-1, -1, 1, 1, -1, -1)), (67, (1, 1, -1, -1, 1, 1))])
def test_terms(n1, bc, n3):
    N = (n1, 8 + n3 % 4, n3)
    oc, gc = O.OracleCase(N, bc, (1.0, 1.0, 1.0), (0.0, 0.0, 0.0)), ih.Case(N, bc)
    rng = np.random.default_rng(11)
    vel, work, nl = (np.ascontiguousarray(rng.standard_normal((3,) + oc.shape)) for _ in range(3))
    for q in range(3):
        gc.upload(ih.VEL1 + q, vel[q])
        gc.upload(ih.WORK1 + q, work[q])
        gc.upload(ih.NL1 + q, nl[q])
    oc.nonlinear(vel, work, nl, oc.zeros())
    oc.helmholtz(1.0 / 137.0, vel, nl)
    for q in range(3):
        for d in range(3):
            gc.interpolate2_pre_vel(q + 1, ih.WORK1 + d, ih.PP)
            gc.nonlinear_upwind(3 * q + d + 1, ih.PP, ih.VEL1 + q, ih.NL1 + q)
        gc.helmholtz(q + 1, 1.0 / 137.0, ih.VEL1 + q, ih.NL1 + q)
        got = gc.download(ih.NL1 + q)
        assert np.array_equal(got, nl[q]), f"component {q + 1}: {int((got != nl[q]).sum())} values differ"
    gc.close()
