"""Where two JOR sweeps are one launch: rows of which four fit 512 threads at every
size, longer ones where the grid is large and the blocks' useful share is, or where a
sweep does not stay in the last-level cache.  The route (the pair's benchmark entry is
refused where the pair is not taken) on both sides of each line; and the values of
long rows on the grids that take the pair, against single sweeps (two calls of one
sweep; a batch that a row past every limit keeps on single sweeps).  Tolerance: none."""
import numpy as np
import pytest

import impact_hip as ih

pytestmark = pytest.mark.gpu

W6, PX, PY = (1,) * 6, (-1, -1, 1, 1, 1, 1), (1, 1, -1, -1, 1, 1)


def takes(c, name):
    ms = ih.C.c_double(0.0)
    rc = c.lib.ih_bench_kernel(c.h, name.encode(), 1, ih.C.byref(ms))
    assert rc in (0, -22)
    return rc == 0


@pytest.mark.parametrize("N,fp64,fp32", [
    ((249, 9, 9), True, True), ((251, 9, 9), False, True), ((499, 9, 9), False, True), ((501, 9, 9), False, False),
    ((270, 60, 61), False, True), ((270, 62, 61), True, True),          # 24 MB in FP64
    ((434, 65, 65), True, True), ((435, 65, 65), False, True),          # the share in FP64
    ((450, 149, 149), False, True), ((450, 150, 149), True, True),      # 240 MB in FP64
    ((505, 62, 62), False, False), ((505, 65, 62), False, True),        # 24 MB in FP32
    ((600, 65, 65), False, True), ((601, 65, 65), False, False),        # the share in FP32
    ((1000, 200, 99), False, False), ((1000, 200, 101), False, True),   # 240 MB in FP32
    ((1013, 200, 101), False, False)],
    ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else None)
def test_route(N, fp64, fp32):
    c = ih.Case(N, W6)
    assert (takes(c, "jor_pair"), takes(c, "jor_pair_f32")) == (fp64, fp32)
    c.close()


@pytest.mark.parametrize("N,bc", [((270, 62, 61), PY), ((434, 65, 65), W6), ((432, 70, 67), PX), ((505, 201, 101), PY),
                                  ((506, 150, 133), W6), ((505, 150, 135), PX)], ids=lambda v: "x".join(map(str, v)))
def test_long_rows_fp64(N, bc):
    c = ih.Case(N, bc, (2.0, 1.0, 1.0))
    assert takes(c, "jor_pair")
    rng = np.random.default_rng(18)
    rel, bb = rng.standard_normal(c.shape), rng.standard_normal(c.shape)
    c.upload(ih.RES, bb)
    last = [N[d] - (bc[2 * d] < 0) for d in range(3)]
    out = []
    for calls in ((5,), (1,) * 5):
        c.upload(ih.PRE, rel)
        for n in calls:
            c.jor(n, 0.8, (1, 1, 1), last)
        out.append(c.download(ih.PRE))
    assert np.array_equal(*out), f"{int((out[0] != out[1]).sum())} values differ"
    c.close()


@pytest.mark.parametrize("N,bc", [((505, 65, 65), PY), ((600, 65, 65), W6), ((601, 70, 67), PX), ((1000, 200, 101), PY),
                                  ((1012, 190, 105), W6)], ids=lambda v: "x".join(map(str, v)))
def test_long_rows_fp32(N, bc):
    p = ih.StepParams(Re=100.0, dtime=1e-4, jor_sweeps=2, jor_omega=0.8, bicg_rel_tol=1e-12, bicg_max_it=2,
                      level_pressure=1, jor_fp32=1, precond_sweeps=4)
    alone, other, row = ih.Case(N, bc, (2.0, 1.0, 1.0)), ih.Case(N, bc, (2.0, 1.0, 1.0)), ih.Case((1100, 8, 9), W6)
    assert takes(alone, "jor_pair_f32") and not takes(row, "jor_pair_f32")
    rng = np.random.default_rng(19)
    for f in (ih.VEL1, ih.VEL2, ih.VEL3):
        v = 0.01 * rng.standard_normal(alone.shape)
        alone.upload(f, v)
        other.upload(f, v)
    ss = alone.timestep(p, 0.0)
    bt = ih.Batch([other, row])
    sb = bt.timestep(p, 0.0)
    assert list(sb[0].bicg_final) == list(ss.bicg_final) and np.all(np.isfinite(list(ss.bicg_final)))
    for f in (ih.PRE, ih.VEL1):
        a, b = alone.download(f), other.download(f)
        assert np.array_equal(a, b), f"field {f}: {int((a != b).sum())} values differ"
    bt.close()
    for c in (alone, other, row):
        c.close()
