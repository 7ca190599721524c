"""Multigrid cycles on thin grids, whose levels have two to five points along one
direction and are too large for the workgroup that runs the coarse levels: the
sweeps, transfers and edge averages of such levels are launches.  Along a periodic
x the row of a level may fit one vector of the sweeps, whose outer neighbours are
then both in that vector.  Tolerance: none, every value is formed as the oracle's
cycle forms it (FP64 and FP32, bit for bit)."""
import numpy as np
import pytest

import impact_hip as ih
import oracle_lib as O

pytestmark = pytest.mark.gpu

W6, PX, PY, PXZ = (1,) * 6, (-1, -1, 1, 1, 1, 1), (1, 1, -1, -1, 1, 1), (-1, -1, 1, 1, -1, -1)
PZ, PXYZ = (1, 1, 1, 1, -1, -1), (-1,) * 6
THIN = [((9, 97, 97), PX),      # FP32: 5 x 49 x 49, four points of the range a row
        ((9, 193, 193), PX),    # FP64 too: 3 x 49 x 49, two points a row
        ((17, 129, 129), PXZ),  # 5 x 33 x 33
        ((9, 129, 161), W6), ((9, 257, 129), PXZ), ((129, 9, 129), PY), ((129, 129, 9), W6),
        ((257, 257, 9), PZ),    # 65 x 65 x 3, two planes
        ((257, 9, 129), PXYZ), ((9, 129, 161), PXYZ)]


@pytest.mark.parametrize("fp32", [False, True], ids=["fp64", "fp32"])
@pytest.mark.parametrize("spec", THIN, ids=lambda s: "x".join(map(str, s[0])) + "-" + "".join("wp"[b < 0] for b in s[1][::2]))
def test_cycle(spec, fp32):
    N, bc = spec
    st = tuple(0.0 if bc[2 * d] < 0 else 1.3 for d in range(3))
    oc, gc = O.OracleCase(N, bc, (2.0, 1.0, 1.0), st), ih.Case(N, bc, (2.0, 1.0, 1.0), st)
    s = tuple(slice(oc.Sp[d] + 3, oc.Np[d] + 4) for d in (2, 1, 0))
    rng = np.random.default_rng(13)
    for cfg in ((15, 4, 4, 4), (15, 3, 2, 1)):
        om = O.OracleMG(oc, *cfg)
        gc.mg_configure(*cfg)
        bb, z = oc.zeros(), rng.standard_normal(oc.shape)
        bb[s] = rng.standard_normal(oc.shape)[s]
        gc.upload(ih.RES, bb)
        gc.upload(ih.PRE, z)
        (om.vcycle_f32 if fp32 else om.vcycle)(bb, z)
        (gc.multigrid_v_f32 if fp32 else gc.multigrid_v)(ih.RES, ih.PRE)
        for f, want, what in ((ih.PRE, z, "result"), (ih.RES, bb, "right-hand side after the averages")):
            got = gc.download(f)[s]
            assert np.array_equal(got, want[s]), f"{what}, cycle {cfg}: {int((got != want[s]).sum())} values differ"
    gc.close()
