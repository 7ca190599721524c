"""Ghost points past a wall whose values are not finite: their coefficients are zero,
and zero times them reaches the wall point in every direction, in the pairs of sweeps
as in single ones and in the oracle (0 * inf and 0 * nan are nan).  Stretches of a
plane that start and end at the first and the last row, and rows of one and several
stretches.  Tolerance: none, the same points are nan and the others are the oracle's
bit for bit."""
import numpy as np
import pytest

import impact_hip as ih
import oracle_lib as O

pytestmark = pytest.mark.gpu

W6, PX, PZ = (1,) * 6, (-1, -1, 1, 1, 1, 1), (1, 1, 1, 1, -1, -1)


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("N,bc", [((8, 9, 10), W6), ((33, 17, 17), W6), ((41, 70, 9), PZ), ((121, 12, 11), W6),
                                  ((300, 40, 10), PX)])
def test_sweeps_beside_ghosts_that_are_not_finite(N, bc, value):
    st = tuple(0.0 if bc[2 * d] < 0 else 1.3 for d in range(3))
    oc, gc = O.OracleCase(N, bc, (2.0, 1.0, 1.0), st), ih.Case(N, bc, (2.0, 1.0, 1.0), st)
    s = tuple(slice(oc.Sp[d] + 3, oc.Np[d] + 4) for d in (2, 1, 0))
    rng = np.random.default_rng(15)
    bb, start = rng.standard_normal(oc.shape), rng.standard_normal(oc.shape)
    gc.upload(ih.RES, bb)
    for d in range(3):
        for side in (0, 1):
            if bc[2 * d + side] < 0:
                continue
            at = [int(rng.integers(1, N[e])) for e in range(3)]  # beside a point of the range
            at[d] = N[d] + 1 if side else 0
            for sweeps in (1, 2, 3, 5):
                rel = start.copy()
                rel[at[2] + 3, at[1] + 3, at[0] + 3] = value
                gc.upload(ih.PRE, rel)
                gc.fill(ih.COMP, 0.0)
                oc.jor(sweeps, 0.8, oc.Sp, oc.Np, rel, bb, oc.zeros())
                gc.jor(sweeps, 0.8, oc.Sp, oc.Np)
                got, want = gc.download(ih.PRE)[s], rel[s]
                assert np.isnan(want).any()
                assert np.array_equal(got, want, equal_nan=True), \
                    f"ghost past side {side} of direction {d + 1}, {sweeps} sweeps: nan at {int(np.isnan(got).sum())}, " \
                    f"oracle {int(np.isnan(want).sum())}"
    gc.close()
