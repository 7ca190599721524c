"""Two JOR sweeps in one launch: rows whose vector count is at the limits of a
block (64, 128 and 256 entries a row with the halo, in FP64 at 122, 250 and 506
points, in FP32 at 244, 500 and 1012), stretches of a plane that end inside a
row, periodic directions down to the fewest points, and the ranges that keep the
single sweeps.  Tolerance: none, the pair forms each value with the operands and
in the order of two single sweeps, which are the oracle's (bit for bit)."""
import ctypes

import numpy as np
import pytest

import impact_hip as ih
import oracle_lib as O
from test_gpu_set_coeffs import SETS

pytestmark = pytest.mark.gpu

W6 = (1, 1, 1, 1, 1, 1)
PY, PZ, PYZ, PX = (1, 1, -1, -1, 1, 1), (1, 1, 1, 1, -1, -1), (1, 1, -1, -1, -1, -1), (-1, -1, 1, 1, -1, -1)
PXY, PXYZ = (-1, -1, -1, -1, 1, 1), (-1,) * 6
# (sizes, boundaries): x lengths on both sides of each limit
PAIRS = [((nx, 9 + nx % 4, 10), bc) for nx, bc in
         [(8, W6), (9, PYZ), (10, PY), (121, W6), (122, PY), (123, PZ), (124, W6), (243, PY), (244, W6), (245, PYZ),
          (249, W6), (250, PYZ), (251, W6), (499, W6), (501, PY), (505, W6), (507, PYZ), (509, W6), (1011, PY),
          (1013, W6), (1018, W6)]]
PAIRS += [((33, 8, 8), PYZ), ((41, 70, 9), PY), ((65, 33, 67), W6), ((34, 37, 131), PZ), ((66, 30, 20), PX)]
PAIRS += [((nx, 9 + nx % 3, 11), bc) for nx, bc in
          [(8, PX), (9, PXYZ), (10, PXY), (11, PX), (65, PXYZ), (122, PXY), (123, PX), (246, PX), (247, PXYZ), (502, PX),
           (506, PX), (507, PXY), (1014, PX), (1020, PX)]]


def same(a, b, what):
    assert np.array_equal(a, b), f"{what}: {int((a != b).sum())} values differ"


@pytest.mark.parametrize("spec", PAIRS, ids=lambda s: "x".join(map(str, s[0])) + "-" + "".join("wp"[b < 0] for b in s[1][::2]))
def test_pairs_of_sweeps(spec):
    N, bc = spec
    st = tuple(0.0 if bc[2 * d] < 0 else 1.3 for d in range(3))
    oc, gc = O.OracleCase(N, bc, (2.0, 1.0, 1.0), st), ih.Case(N, bc, (2.0, 1.0, 1.0), st)
    rng = np.random.default_rng(5)
    rel, bb, phi = (rng.standard_normal(oc.shape) for _ in range(3))
    s = tuple(slice(oc.Sp[d] + 3, oc.Np[d] + 4) for d in (2, 1, 0))
    gc.upload(ih.PRE, rel)
    gc.upload(ih.RES, bb)
    for sweeps in (2, 5):
        oc.jor(sweeps, 0.8, oc.Sp, oc.Np, rel, bb, oc.zeros())
        gc.jor(sweeps, 0.8, oc.Sp, oc.Np)
        same(gc.download(ih.PRE)[s], rel[s], f"{sweeps} FP64 sweeps")
    # the sweeps as M: FP32 from the second on, the last pair writing FP64
    for sweeps in (3, 4):
        p = phi.copy()
        gc.upload(ih.PRE, p)
        oc.bicgstab_mixed(0.0, 1, oc.Sp, oc.Np, bb.copy(), p, sweeps)
        gc.bicgstab_mixed(0.0, 1, oc.Sp, oc.Np, sweeps)
        same(gc.download(ih.PRE)[s], p[s], f"M of {sweeps} FP32 sweeps")
        p = phi.copy()
        gc.upload(ih.PRE, p)
        oc.bicgstab_jor64(0.0, 1, oc.Sp, oc.Np, bb.copy(), p, sweeps)
        gc.bicgstab_jor64(0.0, 1, oc.Sp, oc.Np, sweeps)
        same(gc.download(ih.PRE)[s], p[s], f"M of {sweeps} FP64 sweeps")
    gc.close()


def test_coupling_past_a_wall_keeps_single_sweeps():
    """Uploaded tables that couple the outermost points to the ghost points: two
    sweeps in one call read them as two calls do."""
    spec = ((33, 17, 17), W6, (2.0, 1.0, 1.0), (0.0, 1.5, 1.5))
    oc, gc = O.OracleCase(*spec), ih.Case(*spec, generate=False)
    keep, cs = {}, ih.CoeffSet()
    for field, names in SETS.items():
        for d, name in enumerate(names):
            keep[name] = np.array(oc.coeff(name))
            if name == "cdg2":
                keep[name].reshape(-1)[0] = 0.25 * np.abs(keep[name]).max()
            getattr(cs, field)[d] = keep[name].ctypes.data_as(ctypes.POINTER(ctypes.c_double))
    ih.check(gc.lib.ih_case_set_coeffs(gc.h, ctypes.byref(cs)), "set_coeffs")
    rng = np.random.default_rng(6)
    rel, bb = rng.standard_normal(oc.shape), rng.standard_normal(oc.shape)
    gc.upload(ih.RES, bb)
    out = []
    for calls in ((2,), (1, 1)):
        gc.upload(ih.PRE, rel)
        gc.upload(ih.COMP, rel)
        for n in calls:
            gc.jor(n, 0.8, oc.Sp, oc.Np)
        out.append(gc.download(ih.PRE))
    same(out[0], out[1], "coupled walls")
    gc.close()


@pytest.mark.parametrize("sweeps", [3, 4, 7])
@pytest.mark.parametrize("bcs", [(W6, PZ, W6, PY), (PX, W6, PXY, PZ), (W6, PX, W6)],
                         ids=["walls-and-yz", "periodic-x", "a-row-too-long"])
def test_pairs_in_a_batch(sweeps, bcs):
    """M's FP32 sweeps of several cases in shared launches: each case as alone.  A
    batch with a row past the limit (1100 points) keeps the single sweeps."""
    sizes = [(41, 17, 33), (130, 19, 18), (246, 9, 15), (17, 33, 9)] if len(bcs) == 4 else [(33, 9, 17), (20, 11, 9), (1100, 8, 9)]
    p = ih.StepParams(Re=100.0, dtime=1e-4, jor_sweeps=4, jor_omega=0.8, bicg_rel_tol=1e-12, bicg_max_it=3,
                      level_pressure=1, jor_fp32=1, precond_sweeps=sweeps)
    cases = [[ih.Case(N, bc, (2.0, 1.0, 1.0)) for N, bc in zip(sizes, bcs)] for _ in range(2)]
    for cs in cases:
        rng = np.random.default_rng(10)
        for c in cs:
            for f in (ih.VEL1, ih.VEL2, ih.VEL3):
                c.upload(f, 0.01 * rng.standard_normal(c.shape))
    bt = ih.Batch(cases[0])
    sb = bt.timestep(p, 0.0)
    for q, (a, c) in enumerate(zip(*cases)):
        ss = c.timestep(p, 0.0)
        assert list(sb[q].bicg_final) == list(ss.bicg_final) and np.all(np.isfinite(list(ss.bicg_final))), q
        for f in (ih.PRE, ih.VEL1, ih.VEL2, ih.VEL3):
            same(a.download(f), c.download(f), f"case {q}, field {f}")
    bt.close()
    for c in cases[0] + cases[1]:
        c.close()
