"""The two forms of the fused Poisson operator, chosen by the number of 16 x 16 x
chunk tiles (teams up to 512, one thread per column beyond), at the switch and
at remainders of the tile: one application, and three BiCGstab iterations, which
run the operator with each of its fused dot products.  Tolerance: none, both
forms evaluate the oracle's operations in its order (bit for bit)."""
import numpy as np
import pytest

import impact_hip as ih
import oracle_lib as O

pytestmark = pytest.mark.gpu

W6 = (1, 1, 1, 1, 1, 1)
FORMS = [
    pytest.param(((2048, 17, 33), W6), id="512-tiles-teams"),           # 128 x 2 x 2, one row and one plane over
    pytest.param(((2049, 17, 33), W6), id="516-tiles-column"),          # and one column over
    pytest.param(((2050, 16, 34), (-1, -1, 1, 1, -1, -1)), id="periodic-xz-column"),
    pytest.param(((530, 31, 129), (1, 1, -1, -1, 1, 1)), id="periodic-y-teams"),  # 34 x 2 x 5
    pytest.param(((9, 9, 9), W6), id="one-tile"),
]


def same(a, b, what):
    assert np.array_equal(a, b), f"{what}: {int((a != b).sum())} values differ"


@pytest.mark.parametrize("spec", FORMS)
def test_operator_and_its_dots(spec):
    N, bc = spec
    oc, gc = O.OracleCase(N, bc, (1.0, 1.0, 1.0), (0.0, 0.0, 0.0)), ih.Case(N, bc)
    rng = np.random.default_rng(3)
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
