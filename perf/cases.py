"""The work that users of this library have it do, as cases to be timed.

A case is a dict of plain values: a kind of call, a grid and its options.
listed() names a fixed set, draw() gives more of the same ranges.  prepare()
builds what a program has in hand before the call (a resident ih.Case with its
coefficients, or a batch of them, inputs and result buffers on the host), run()
makes the calls through the Python mirror of the C ABI and returns the fields
that they compute, work() counts what a pass cannot do without, and exact()
evaluates the cases that have a closed numpy/torch form in float64.

Fields cross the boundary as arrays in the library's layout, which is how every
host program of this library gets at its results, so a pass ends with the
download of what it computed into page-locked arrays that the state owns.
"""
import ctypes
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "gpu-impact-ct_amd"))
import impact_hip as ih  # noqa: E402

WALLS = "wwwwww"  # lower and upper condition of x, y, z: w wall, p periodic
TUBE_L, TUBE_STRETCH = (2.0, 1.0, 1.0), (0.0, 1.5, 1.5)


def listed():
    return [
        # A host program's own call of the drop-in Jacobi solver on its arrays: the smallest grid of the tests.
        {"name": "jacobi_dropin_33x17x17", "kind": "jacobi", "n1": 33, "n2": 17, "n3": 17, "bc": WALLS},
        # A Poisson solve to convergence on a grid of a few thousand points: launches and latency alone.
        {"name": "solve_33x17x17", "kind": "solve", "n1": 33, "n2": 17, "n3": 17, "bc": WALLS, "form": "fp64",
         "iterations": 400},
        # The momentum terms of one substep, call by call, as a host that keeps its own time loop makes them.
        {"name": "momentum_129x65x65", "kind": "momentum", "n1": 129, "n2": 65, "n3": 65, "bc": WALLS},
        # The reference's GPU path in itself: 200 Jacobi over-relaxation sweeps on the benchmark grid.
        {"name": "relax_257x129x129", "kind": "relax", "n1": 257, "n2": 129, "n3": 129, "bc": WALLS, "sweeps": 200},
        # One time step of the 64^3-cell channel, the smallest whole run of the benchmark.
        {"name": "step_channel_65", "kind": "step", "n1": 65, "n2": 65, "n3": 65, "bc": WALLS, "form": "fp64"},
        # One time step of a channel periodic in x and z on a ragged grid (no size a multiple of any tile).
        {"name": "step_duct_118x71x91", "kind": "step", "n1": 118, "n2": 71, "n3": 91, "bc": "ppwwpp", "form": "fp64"},
        # A served request's step: 96^3 cells with the reference's multigrid preconditioner.
        {"name": "step_multigrid_97", "kind": "step", "n1": 97, "n2": 97, "n3": 97, "bc": WALLS, "form": "multigrid"},
        # The benchmark's own step in its three forms: plain FP64, FP32-preconditioned, multigrid.
        {"name": "step_tube_257", "kind": "step", "n1": 257, "n2": 129, "n3": 129, "bc": WALLS, "form": "fp64"},
        {"name": "step_tube_257_mixed", "kind": "step", "n1": 257, "n2": 129, "n3": 129, "bc": WALLS, "form": "mixed"},
        {"name": "step_tube_257_multigrid", "kind": "step", "n1": 257, "n2": 129, "n3": 129, "bc": WALLS,
         "form": "multigrid"},
        # Six patients' tubes of uneven size advanced together.
        {"name": "batch_6_tubes", "kind": "batch", "cases": 6, "sizes": 0, "sweeps": 8},
        # The largest grid of the benchmark, past the last-level cache: a bounded number of BiCGstab iterations.
        {"name": "solve_385x193x193", "kind": "solve", "n1": 385, "n2": 193, "n3": 193, "bc": WALLS, "form": "fp64",
         "iterations": 40},
    ]


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _bc(rng, flow):
    """Conditions of a box: of a flow (walls, a duct, a channel), or any for the calls that need no such flow."""
    return rng.choice([WALLS, WALLS, WALLS, "wwwwpp", "ppwwpp"] + ([] if flow else ["wwppww", "pppppp"]))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "solve", "relax", "momentum", "jacobi", "batch"])
    if kind == "step":
        form = rng.choice(["fp64", "mixed", "multigrid"])
        if form == "multigrid":  # sizes that halve at least three times
            n = [8 * _size(rng, 2, 24) + 1 for _ in range(3)]
            return {"kind": kind, "n1": n[0], "n2": n[1], "n3": n[2], "bc": WALLS, "form": form}
        n = [_size(rng, 17, 160) for _ in range(3)]
        return {"kind": kind, "n1": n[0], "n2": n[1], "n3": n[2], "bc": _bc(rng, True), "form": form}
    if kind == "solve":
        n = [_size(rng, 17, 257) for _ in range(3)]
        return {"kind": kind, "n1": n[0], "n2": n[1], "n3": n[2], "bc": _bc(rng, True),
                "form": rng.choice(["fp64", "mixed"]), "iterations": rng.randrange(20, 81)}
    if kind == "relax":
        n = [_size(rng, 17, 300) for _ in range(3)]
        return {"kind": kind, "n1": n[0], "n2": n[1], "n3": n[2], "bc": _bc(rng, False), "sweeps": rng.randrange(50, 251)}
    if kind == "batch":
        return {"kind": kind, "cases": rng.randrange(2, 7), "sizes": rng.randrange(1, 1000),
                "sweeps": rng.choice([2, 4, 8, 16])}
    n = [_size(rng, 13, 200 if kind == "momentum" else 80) for _ in range(3)]
    return {"kind": kind, "n1": n[0], "n2": n[1], "n3": n[2], "bc": _bc(rng, False)}


# ---- grids -----------------------------------------------------------------------------------------------------
def _grid(case):
    return case["n1"], case["n2"], case["n3"]


def _bcs(case):
    return tuple(-1 if ch == "p" else 1 for ch in case["bc"])


def _shape(case):
    """(lengths, stretching): the tube's for a step on a walled box longer than wide, else a unit box's."""
    n, walls = _grid(case), case["bc"] == WALLS
    if case["kind"] in ("step", "solve", "relax") and walls and n[0] > 1.5 * n[1] and min(n[1:]) >= 17:
        return TUBE_L, TUBE_STRETCH
    return (1.0, 1.0, 1.0), (0.0, 0.0, 0.0)


BATCH_SIZES = ((65, 65, 65), (97, 97, 97), (129, 65, 65), (193, 97, 97))  # the benchmark's


def _batch_grids(case):
    """The grids of a batch: the benchmark's four sizes in turn, or drawn from them by the case's own number."""
    if case["sizes"] == 0:
        return [BATCH_SIZES[q % 4] for q in range(case["cases"])]
    pick = np.random.default_rng(case["sizes"])
    return [BATCH_SIZES[int(pick.integers(3))] for _ in range(case["cases"])]


def _radius(x, radius, stenosis):
    delta = 1.0 - math.sqrt(1.0 - stenosis)
    r = np.full_like(x, radius)
    s = np.abs(x - 1.0) <= 0.4
    r[s] = radius * (1.0 - delta / 2.0 * (1.0 + np.cos(np.pi * (x[s] - 1.0) / 0.4)))
    return r


# ---- inputs ----------------------------------------------------------------------------------------------------
def _rng(seed):
    return np.random.default_rng([int(seed), 20240])


def _smooth(rng, shape, amplitude):
    """A field of a few long waves with a little noise, as flow fields have."""
    z, y, x = np.meshgrid(*[np.linspace(0.0, 1.0, n) for n in shape], indexing="ij", sparse=True)
    f = np.zeros(shape)
    for _ in range(3):
        kx, ky, kz = rng.integers(1, 4, 3)
        a, b, c = rng.uniform(0.0, 2.0 * np.pi, 3)
        f += np.sin(2 * np.pi * kx * x + a) * np.sin(2 * np.pi * ky * y + b) * np.sin(2 * np.pi * kz * z + c)
    return amplitude * (f / 3.0 + 0.01 * rng.standard_normal(shape))


def _pinned(shape):
    if torch.cuda.is_available():
        return torch.zeros(shape, dtype=torch.float64, pin_memory=True).numpy()
    return np.zeros(shape)


def _new_case(case, seed):
    L, st = _shape(case)
    return ih.Case(_grid(case), _bcs(case), L, st, device=0)


def _params(form, sweeps=16, tube=True):
    return ih.StepParams(Re=500.0 if tube else 100.0, dtime=5e-4 if tube else 1e-3, jor_sweeps=200, jor_omega=0.8,
                         bicg_rel_tol=1e-8, bicg_max_it=2000, level_pressure=1, inflow_kind=2 if tube else 1,
                         inflow_amp=1.0, use_mask=1 if tube else 0, jor_fp32=1 if form == "mixed" else 0,
                         precond_sweeps=sweeps if form == "mixed" else 0,
                         precond_poisson=1 if form == "multigrid" else 0)


def _flow(c, rng, tube):
    """Three velocity components: plug flow in the tube's lumen, or a channel profile, with a disturbance."""
    vel = [_smooth(rng, c.shape, 0.05) for _ in range(3)]
    if tube:
        radius, stenosis = float(rng.uniform(0.2, 0.35)), float(rng.uniform(0.3, 0.7))
        c.set_tube_mask(0.5, 0.5, _radius(c.coords(0, 1), radius, stenosis), _radius(c.coords(0, 0), radius, stenosis))
        m = c.get_mask()
        vel = [(v + (1.0 if q == 0 else 0.0)) * m[q] for q, v in enumerate(vel)]
    else:
        y, z = np.linspace(0, 1, c.shape[1])[None, :, None], np.linspace(0, 1, c.shape[0])[:, None, None]
        vel[0] += 16.0 * y * (1.0 - y) * z * (1.0 - z)
    out = []
    for v in vel:
        p = _pinned(c.shape)
        p[...] = v
        out.append(p)
    return out


class State:
    def __init__(self, kind):
        self.kind = kind


def prepare(case, seed):
    rng = _rng(seed)
    s = State(case["kind"])
    if s.kind == "batch":
        s.cases = [ih.Case(n, (1,) * 6, TUBE_L, TUBE_STRETCH, device=0) for n in _batch_grids(case)]
        s.vel = [_flow(c, rng, True) for c in s.cases]
        s.out = [[_pinned(c.shape) for _ in range(4)] for c in s.cases]
        s.batch = ih.Batch(s.cases)
        s.params = _params("mixed", case["sweeps"])
        return s
    c = s.case = _new_case(case, seed)
    if s.kind == "step":
        tube = _shape(case)[0] == TUBE_L
        s.params = _params(case["form"], tube=tube)
        s.vel = _flow(c, rng, tube)
        s.out = [_pinned(c.shape) for _ in range(4)]
    elif s.kind == "solve":
        # the right-hand side a step has: the divergence of a disturbed velocity
        for q in range(3):
            c.upload(ih.VEL1 + q, _smooth(rng, c.shape, 1.0))
        c.divergence2()
        s.form, s.iterations = case["form"], case["iterations"]
        s.eps = 1e-8 * float(np.abs(_inner(c, c.download(ih.RES))).max())
        s.out = [_pinned(c.shape)]
    elif s.kind == "relax":
        c.upload(ih.RES, _smooth(rng, c.shape, 1.0))
        s.sweeps = case["sweeps"]
        s.out = [_pinned(c.shape)]
    elif s.kind == "momentum":
        for q in range(3):
            c.upload(ih.VEL1 + q, _smooth(rng, c.shape, 1.0))
        s.out = [_pinned(c.shape) for _ in range(4)]
    elif s.kind == "jacobi":
        s.guess, s.rhs, s.rel = _smooth(rng, c.shape, 0.01), _smooth(rng, c.shape, 1.0), np.zeros(c.shape)
    return s


def _inner(c, a, q=None, interior=False):
    """The part of a field that the library computes: the pressure range, or a velocity component's."""
    lo, hi = (c.Sp, c.Np) if q is None else (c.SI[q], c.NI[q]) if interior else (c.SB[q], c.NB[q])
    return a[tuple(slice(lo[d] + 3, hi[d] + 4) for d in (2, 1, 0))]


def _download(c, f, a):
    ih.check(c.lib.ih_field_download(c.h, f, a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))), "download")
    return a


def _start(c, vel):
    for q in range(3):
        c.upload(ih.VEL1 + q, vel[q])
    c.fill(ih.PRE, 0.0)


def _result(c, out):
    for q in range(3):
        _download(c, ih.VEL1 + q, out[q])
    _download(c, ih.PRE, out[3])
    return [_inner(c, out[q], q) for q in range(3)] + [_inner(c, out[3])]


def run(s):
    if s.kind == "batch":
        for c, vel in zip(s.cases, s.vel):
            _start(c, vel)
        s.batch.timestep(s.params, 0.0, stats=False)
        return [_result(c, out) for c, out in zip(s.cases, s.out)]
    c = s.case
    if s.kind == "step":
        _start(c, s.vel)
        c.timestep(s.params, 0.0, stats=False)
        return _result(c, s.out)
    if s.kind == "solve":
        c.fill(ih.PRE, 0.0)
        if s.form == "mixed":
            st = c.bicgstab_mixed(s.eps, s.iterations, c.Sp, c.Np, 16)
        else:
            st = c.bicgstab(s.eps, s.iterations, c.Sp, c.Np)
        return [_inner(c, _download(c, ih.PRE, s.out[0])), st.iterations]
    if s.kind == "relax":
        c.fill(ih.PRE, 0.0)
        c.jor(s.sweeps, 0.8, c.Sp, c.Np)
        return [_inner(c, _download(c, ih.PRE, s.out[0]))]
    if s.kind == "momentum":
        for d in (1, 2, 3):
            for q in (1, 2, 3):
                c.exchange(d, q, ih.VEL1 + q - 1)
        c.interpolate_vel()
        for q in range(3):
            for d in range(3):
                c.interpolate2_pre_vel(q + 1, ih.WORK1 + d, ih.PP)
                c.nonlinear_upwind(3 * q + d + 1, ih.PP, ih.VEL1 + q, ih.NL1 + q)
            c.helmholtz(q + 1, 1.0 / 500.0, ih.VEL1 + q, ih.NL1 + q)
        c.divergence2()
        for q in range(3):
            _download(c, ih.NL1 + q, s.out[q])
        _download(c, ih.RES, s.out[3])
        return [_inner(c, s.out[q], q, True) for q in range(3)] + [_inner(c, s.out[3])]
    np.copyto(s.rel, s.guess)
    c.device_jacobi_solver(0.8, c.Sp, c.Np, s.rel, s.rhs)
    return [_inner(c, s.rel)]


# ---- what a pass cannot do without -----------------------------------------------------------------------------
# floating-point operations a point: the substep's stencils, a sweep, a BiCGstab iteration with two operators
STENCILS, SWEEP, ITERATION = 420, 17, 2 * 70 + 22
ITERATIONS = {"fp64": 900, "mixed": 160, "multigrid": 60}  # of one solve to 1e-8 on the benchmark grid


def _step_flops(form, sweeps=16):
    m = {"fp64": 0, "mixed": 2 * sweeps * SWEEP, "multigrid": 2 * 1.3 * 9 * SWEEP}[form]
    return 3 * (STENCILS + 200 * SWEEP + ITERATIONS[form] * (ITERATION + m))


def work(case):
    kind = case["kind"]
    if kind == "batch":
        points = sum(math.prod(n) for n in _batch_grids(case))
        return {"bytes": 7 * 8 * points, "flops": points * _step_flops("mixed", case["sweeps"])}
    points = math.prod(_grid(case))
    if kind == "step":
        return {"bytes": 7 * 8 * points, "flops": points * _step_flops(case["form"])}
    if kind == "solve":
        m = 2 * 16 * SWEEP if case["form"] == "mixed" else 0
        return {"bytes": 2 * 8 * points, "flops": points * case["iterations"] * (ITERATION + m)}
    if kind == "relax":
        return {"bytes": 2 * 8 * points, "flops": points * case["sweeps"] * SWEEP}
    if kind == "momentum":
        return {"bytes": 7 * 8 * points, "flops": points * (3 * 3 * 26 + 3 * 43 + 3 * 11 + 33)}
    return {"bytes": 3 * 8 * points, "flops": points * 40 * SWEEP}


# ---- the cases with a closed form, in float64 without the library ----------------------------------------------
def _coordinates(n, length, factor, periodic):
    """Pressure and velocity coordinates of one direction at -3..n+3, element i at [i + 3]."""
    def at(t):
        s = (t - 1.0) / (n - 1.0)
        if factor == 0.0:
            return s * length
        top = math.tanh(factor)
        return length * (math.atanh(top * (2.0 * s - 1.0)) / factor + 1.0) / 2.0

    p, u = np.zeros(n + 7), np.zeros(n + 7)
    for i in range(1, n + 1):
        p[i + 3] = at(i)
    for i in range(0, n + 1):
        u[i + 3] = at(i + 0.5)
    for i in range(-3, n + 4):
        if periodic:
            if i < 1 or i >= n:
                turn = (i - 1) // (n - 1)
                p[i + 3] = p[i - turn * (n - 1) + 3] + turn * length
                u[i + 3] = u[i - turn * (n - 1) + 3] + turn * length
        elif i < 1:
            p[i + 3] = 2 * p[4] - p[2 - i + 3]
            if i < 0:
                u[i + 3] = 2 * p[4] - u[1 - i + 3]
        elif i > n:
            p[i + 3] = 2 * p[n + 3] - p[2 * n - i + 3]
            u[i + 3] = 2 * p[n + 3] - u[2 * n - 1 - i + 3]
    return p, u


def _compact(n, p, u, periodic):
    """The three taps of the compact second difference that the relaxation solves with, rows 1..n."""
    t = np.zeros((n + 1, 3))
    for i in range(1, n + 1):
        low = 0.0 if i == 1 and not periodic else 1.0 / ((u[i + 3] - u[i + 2]) * (p[i + 3] - p[i + 2]))
        high = 0.0 if i == n and not periodic else 1.0 / ((u[i + 3] - u[i + 2]) * (p[i + 4] - p[i + 3]))
        twice = 2.0 if not periodic and i in (1, n) else 1.0
        t[i] = twice * low, -twice * (low + high), twice * high
    return t


def _exact_relax(case, b, sweeps, x):
    n, bc = _grid(case), _bcs(case)
    L, st = _shape(case)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    per = [bc[2 * d] == -1 for d in range(3)]
    hi = [n[d] - 1 if per[d] else n[d] for d in range(3)]
    box = tuple(slice(4, hi[d] + 4) for d in (2, 1, 0))
    b, x = (torch.from_numpy(np.ascontiguousarray(a[box])).to(dev) for a in (b, x))
    taps = []
    for d in range(3):
        t = _compact(n[d], *_coordinates(n[d], L[d], st[d], per[d]), per[d])[1:hi[d] + 1]
        view = [1, 1, 1]
        view[2 - d] = hi[d]
        taps.append([torch.from_numpy(np.ascontiguousarray(t[:, q])).to(dev).reshape(view) for q in range(3)])
    diag = taps[0][1] + taps[1][1] + taps[2][1]
    for _ in range(sweeps):
        s = b.clone()
        for d in range(3):  # the taps over a wall are zero, so the turn of roll() does not matter there
            s -= taps[d][0] * torch.roll(x, 1, 2 - d) + taps[d][2] * torch.roll(x, -1, 2 - d)
        x = 0.8 * s / diag + 0.2 * x
    return [x.cpu().numpy()]


def _weights(offsets, order):
    """Finite-difference weights at 0 of the given derivative for samples at the offsets."""
    a = np.vander(np.asarray(offsets, dtype=np.float64), increasing=True).T
    r = np.zeros(len(offsets))
    r[order] = math.factorial(order)
    return np.linalg.solve(a, r)


def _table(order, bias, widths, x, periodic, shift, first, n):
    """Rows first..n of a stencil table on mapped coordinates, taps -3..3 around the row's index: the order-th
    derivative from `widths` samples (per row from a wall inwards, the last one inside), the window centred and, at a
    wall, moved to lie within the samples.  shift: where a sample of the row's own index lies from it (0, or half a
    cell for tables between the pressure and the velocity points); bias -1 or 1 leaves out the far sample on the
    lower or upper side, which makes an upwind stencil."""
    t = np.zeros((n + 1, 7))
    sample_low = 1 if shift < 0 or (shift == 0 and first == 1) else 0
    for i in range(first, n + 1):
        k = widths[-1] if periodic else widths[min(i - first, n - i, len(widths) - 1)]
        half = k // 2
        right = half if shift < 0 else half - 1 if shift > 0 else (k - 1) // 2
        left = right - k + 1
        if not periodic:
            move = max(sample_low - (i + left), 0) - max(i + right - n, 0)
            left, right = left + move, right + move
        if bias < 0 and (periodic or i - first >= half):
            left += 1
        if bias > 0 and (periodic or n - i >= half):
            right -= 1
        taps = np.arange(left, right + 1)
        at = taps + shift
        w = _weights(at, order)
        if order > 0:
            xs = x[i + taps + 3]
            w1 = _weights(at, 1)
            d1 = w1 @ xs
            w = w1 / d1 if order == 1 else w / d1 ** 2 - w1 * (w @ xs) / d1 ** 3
        t[i, taps + 3] = w
    return t


def _ghosts(f, n, bc, d, vel_dir):
    """The ghost layers of f along d: turned round a period, zero past a wall (a normal component keeps row 0)."""
    axis = 2 - d
    g = np.moveaxis(f, axis, 0)
    if bc[2 * d] == -1:
        for i in list(range(-3, 1)) + list(range(n[d], n[d] + 4)):
            g[i + 3] = g[(i - 1) % (n[d] - 1) + 1 + 3]
    else:
        g[:(3 if vel_dir == d + 1 else 4)] = 0.0
        g[n[d] + 4:] = 0.0


def _along(table, f, d, lo, hi):
    """The stencil table applied along d over the box lo..hi."""
    out = 0.0
    box = [slice(lo[e] + 3, hi[e] + 4) for e in (2, 1, 0)]
    view = [1, 1, 1]
    view[2 - d] = hi[d] - lo[d] + 1
    for tap in range(-3, 4):
        b = list(box)
        b[2 - d] = slice(lo[d] + tap + 3, hi[d] + tap + 4)
        w = table[lo[d]:hi[d] + 1, tap + 3].reshape(view)
        out = out + np.where(w != 0.0, w * f[tuple(b)], 0.0)
    return out


UPWIND, BETWEEN, ONTO = (4, 5, 5, 7), (3, 4, 4, 6), (4, 4, 6, 6)  # stencil widths from a wall inwards


def _exact_momentum(case, vel):
    n, bc = _grid(case), _bcs(case)
    L, st = _shape(case)
    per = [bc[2 * d] == -1 for d in range(3)]
    xs = [_coordinates(n[d], L[d], st[d], per[d]) for d in range(3)]
    sp, np_ = [1] * 3, [n[d] - 1 if per[d] else n[d] for d in range(3)]
    for f, v in enumerate(vel):
        for d in range(3):
            _ghosts(v, n, bc, d, f + 1)
    work = []
    for m in range(3):
        w = np.zeros_like(vel[m])
        box = tuple(slice(4, np_[d] + 4) for d in (2, 1, 0))
        w[box] = _along(_table(0, 0, ONTO, None, per[m], 0.5, 1, n[m]), vel[m], m, sp, np_)
        for d in range(3):
            _ghosts(w, n, bc, d, 0)
        work.append(w)
    out = []
    for q in range(3):
        lo = [1 if per[d] or d == q else 2 for d in range(3)]
        hi = [n[d] - 1 for d in range(3)]
        nl, helm = 0.0, 0.0
        for d in range(3):
            pp = _along(_table(0, 0, BETWEEN, None, per[q], -0.5, 0, n[q]), work[d], q, lo, hi)
            x, first = (xs[d][1], 0) if d == q else (xs[d][0], 1)
            up, down = (_along(_table(1, b, UPWIND, x, per[d], 0, first, n[d]), vel[q], d, lo, hi) for b in (1, -1))
            nl = nl + np.where(pp >= 0.0, up, down) * pp
            helm = helm + _along(_table(2, 0, UPWIND, x, per[d], 0, first, n[d]), vel[q], d, lo, hi)
        out.append(nl - helm / 500.0)
    div = sum(_along(_table(1, 0, ONTO, xs[m][1], per[m], 0.5, 1, n[m]), vel[m], m, sp, np_) for m in range(3))
    return out + [div]


def exact(case, seed):
    n = _grid(case) if "n1" in case else None
    shape = (n[2] + 7, n[1] + 7, n[0] + 7) if n else None
    if case["kind"] == "relax" and math.prod(n) * case["sweeps"] < 2e9:
        return _exact_relax(case, _smooth(_rng(seed), shape, 1.0), case["sweeps"], np.zeros(shape))
    if case["kind"] == "momentum":
        rng = _rng(seed)
        return _exact_momentum(case, [_smooth(rng, shape, 1.0) for _ in range(3)])
    return None  # solves and steps stop by a test on a residual, so their iterates have no such value
