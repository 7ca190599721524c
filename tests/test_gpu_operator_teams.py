"""The operator in two teams a tile with its dot products fused, across a periodic z:
grids whose tiles do not exceed two a compute unit and whose columns leave no room for
short z chunks (171 to 512 columns of one reduction chunk, 86 to 256 of two), at both
ends of each range.  One application, and BiCGstab iterations, which take all of its
dot products.  Tolerance: none, operator and sums are the oracle's operations in their
order (bit for bit)."""
import numpy as np
import pytest

import impact_hip as ih
import oracle_lib as O

pytestmark = pytest.mark.gpu

PZ, PYZ, PXZ, PXYZ = (1, 1, 1, 1, -1, -1), (1, 1, -1, -1, -1, -1), (-1, -1, 1, 1, -1, -1), (-1,) * 6
GRIDS = [((2736, 9, 20), PZ), ((2737, 18, 33), PXYZ),  # 171 and 342 columns, one chunk of 19 and of 32
         ((4096, 17, 9), PZ), ((1370, 16, 41), PYZ),   # 512, one chunk; 86, two chunks
         ((4097, 12, 34), PXZ)]                        # 256, two chunks of 16 and 17


@pytest.mark.parametrize("spec", GRIDS, ids=lambda s: "x".join(map(str, s[0])) + "-" + "".join("wp"[b < 0] for b in s[1][::2]))
def test_operator_and_its_dots(spec):
    N, bc = spec
    oc, gc = O.OracleCase(N, bc, (1.0, 1.0, 1.0), (0.0, 0.0, 0.0)), ih.Case(N, bc)
    rng = np.random.default_rng(22)
    p = rng.standard_normal(oc.shape)
    lap = oc.zeros()
    gc.upload(ih.TMP1, p)
    oc.product_div_grad(p.copy(), lap, oc.zeros())
    gc.product_div_grad(ih.TMP1, ih.TMP2)
    s = tuple(slice(oc.Sp[d] + 3, oc.Np[d] + 4) for d in (2, 1, 0))
    got = gc.download(ih.TMP2)[s]
    assert np.array_equal(got, lap[s]), f"A p: {int((got != lap[s]).sum())} values differ"
    phi = oc.zeros()
    gc.upload(ih.RES, lap)
    for sweeps, its in ((0, 3), (2, 2)):
        gc.upload(ih.PRE, phi)
        if sweeps:
            so, sg = oc.bicgstab_mixed(0.0, its, oc.Sp, oc.Np, lap, phi, sweeps), gc.bicgstab_mixed(0.0, its, oc.Sp, oc.Np, sweeps)
        else:
            so, sg = oc.bicgstab(0.0, its, oc.Sp, oc.Np, lap, phi), gc.bicgstab(0.0, its, oc.Sp, oc.Np)
        assert (so.iterations, so.exit_reason, so.norm_inf_final) == (sg.iterations, sg.exit_reason, sg.norm_inf_final)
        got = gc.download(ih.PRE)[s]
        assert np.array_equal(got, phi[s]), f"{sweeps} sweeps of M: {int((got != phi[s]).sum())} values differ"
    gc.close()
