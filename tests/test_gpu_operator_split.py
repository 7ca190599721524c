"""The operator in short z chunks with its dot products in a launch of their own,
taken where its tiles leave most of the device idle: at the rule's line (three
times as many chunks as the reduction has) and beside it, at remainders of planes,
chunks and tiles.  One application, and BiCGstab iterations, which take all of its
dot products.  Tolerance: none, operator and partial sums are the fused ones' and
the oracle's operations in their order (bit for bit)."""
import numpy as np
import pytest

import impact_hip as ih
import oracle_lib as O

pytestmark = pytest.mark.gpu

W6 = (1, 1, 1, 1, 1, 1)
GRIDS = [((8, 8, 8), W6), ((9, 17, 10), (1, 1, -1, -1, 1, 1)), ((17, 16, 33), W6), ((40, 33, 34), (-1, -1, 1, 1, -1, -1)),
         ((33, 32, 65), (1, 1, 1, 1, -1, -1)), ((272, 80, 64), W6),  # 85 columns: 6 chunks, of 2
         ((273, 80, 64), W6),                                        # 90: 5, fused
         ((61, 47, 95), W6), ((100, 20, 131), (-1,) * 6)]


def same(a, b, what):
    assert np.array_equal(a, b), f"{what}: {int((a != b).sum())} values differ"


@pytest.mark.parametrize("spec", GRIDS, ids=lambda s: "x".join(map(str, s[0])) + "-" + "".join("wp"[b < 0] for b in s[1][::2]))
def test_operator_and_its_dots(spec):
    N, bc = spec
    oc, gc = O.OracleCase(N, bc, (1.0, 1.0, 1.0), (0.0, 0.0, 0.0)), ih.Case(N, bc)
    rng = np.random.default_rng(4)
    p = rng.standard_normal(oc.shape)
    lap = oc.zeros()
    gc.upload(ih.TMP1, p)
    oc.product_div_grad(p.copy(), lap, oc.zeros())
    gc.product_div_grad(ih.TMP1, ih.TMP2)
    s = tuple(slice(oc.Sp[d] + 3, oc.Np[d] + 4) for d in (2, 1, 0))
    same(gc.download(ih.TMP2)[s], lap[s], "A p")
    phi = oc.zeros()
    gc.upload(ih.RES, lap)
    gc.upload(ih.PRE, phi)
    so = oc.bicgstab(0.0, 3, oc.Sp, oc.Np, lap, phi)
    sg = gc.bicgstab(0.0, 3, oc.Sp, oc.Np)
    assert (so.iterations, so.exit_reason, so.norm_inf_final) == (sg.iterations, sg.exit_reason, sg.norm_inf_final)
    same(gc.download(ih.PRE)[s], phi[s], "BiCGstab iterate")
    so = oc.bicgstab_mixed(0.0, 2, oc.Sp, oc.Np, lap, phi, 2)
    sg = gc.bicgstab_mixed(0.0, 2, oc.Sp, oc.Np, 2)
    assert (so.iterations, so.norm_inf_final) == (sg.iterations, sg.norm_inf_final)
    same(gc.download(ih.PRE)[s], phi[s], "preconditioned BiCGstab iterate")
    gc.close()
