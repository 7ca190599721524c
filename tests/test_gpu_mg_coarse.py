"""The multigrid levels that run in one workgroup, and the edge averages that the
transfers between levels form as they read: level sizes on both sides of the
workgroup's limit (3072 points of a level), levels of three points, directions
that stop halving before the others, periodic pairs.  Tolerance: none, every
value is formed as the oracle's cycle forms it (FP64 and FP32, bit for bit)."""
import numpy as np
import pytest

import impact_hip as ih
import oracle_lib as O

pytestmark = pytest.mark.gpu

W6 = (1, 1, 1, 1, 1, 1)
CYCLES = [((9, 9, 9), W6), ((11, 9, 17), (1, 1, -1, -1, 1, 1)), ((27, 27, 27), W6),  # 14^3 = 2744
          ((27, 31, 27), W6), ((29, 29, 27), W6),  # 14 x 16 x 14 = 3136, 15 x 15 x 14 = 3150: launched
          ((33, 25, 27), (-1, -1, 1, 1, 1, 1)),    # 17 x 13 x 14 = 3094, 2912 of its range
          ((65, 9, 9), W6), ((9, 65, 8), W6), ((8, 9, 33), (1, 1, 1, 1, -1, -1)), ((17, 33, 9), (-1, -1, -1, -1, 1, 1)),
          ((49, 25, 41), W6), ((33, 17, 17), (-1, -1, -1, -1, -1, -1))]


@pytest.mark.parametrize("fp32", [False, True], ids=["fp64", "fp32"])
@pytest.mark.parametrize("spec", CYCLES, ids=lambda s: "x".join(map(str, s[0])) + "-" + "".join("wp"[b < 0] for b in s[1][::2]))
def test_cycle(spec, fp32):
    N, bc = spec
    st = tuple(0.0 if bc[2 * d] < 0 else 1.3 for d in range(3))
    oc, gc = O.OracleCase(N, bc, (2.0, 1.0, 1.0), st), ih.Case(N, bc, (2.0, 1.0, 1.0), st)
    s = tuple(slice(oc.Sp[d] + 3, oc.Np[d] + 4) for d in (2, 1, 0))
    rng = np.random.default_rng(9)
    for cfg in ((15, 4, 4, 4), (15, 1, 2, 3)):
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
