"""The single-term momentum calls on both sides of the line between one plane a thread
and several (2048 wavefronts of 64 points at one plane each), with every remainder of
the planes, each component and direction.  Tolerance: none (the oracle's operations in
its order)."""
import numpy as np
import pytest

import impact_hip as ih
import oracle_lib as O

pytestmark = pytest.mark.gpu

W6, PXZ, PY = (1,) * 6, (-1, -1, 1, 1, -1, -1), (1, 1, -1, -1, 1, 1)


@pytest.mark.parametrize("N,bc", [((64, 64, 32), W6), ((64, 65, 33), W6), ((64, 66, 34), PXZ), ((64, 67, 35), PY),
                                  ((66, 120, 9), W6), ((130, 86, 10), PXZ), ((9, 210, 11), PY), ((200, 64, 12), W6),
                                  ((65, 47, 61), PXZ)], ids=lambda v: "x".join(map(str, v)))
def test_terms(N, bc):
    oc, gc = O.OracleCase(N, bc, (1.0, 1.0, 1.0), (0.0, 0.0, 0.0)), ih.Case(N, bc)
    rng = np.random.default_rng(20)
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
