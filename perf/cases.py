"""Performance cases of the multigrid framework: the calls its users make,
through the public entry points (mgp.Solver, mgp.Batch, mgp.Server and the
kernel-level C ABI on caller-owned device arrays), over the range of sizes,
types and face mixes they are made with.

A case is a dict of plain values.  kind says which call it is:

  solve      mgp.Solver.solve from a zero guess on a resident hierarchy
             (FP64, or FP32 cycles inside FP64 refinement)
  vcycles    reference mode, V-cycles with full weighting on Dirichlet faces, a
             fixed number of them (the reference's own way of running)
  batch      mgp.Batch: many small uneven problems solved together
  server     mgp.Server: a burst of requests of mixed shapes and face types
  pair       mgp_rbgs_sweep2_*: a pair of Gauss-Seidel sweeps
  correct    mgp_rbgs_sweep2_prolong_*: the cycle's correction and the pair of
             sweeps after it (the way up)
  descend    mgp_bc_neumann_faces_* and mgp_residual_restrict_fw_*: residual and
             restriction (the way down)
  update     mgp_update_residual_hilo_f64_f32: update and residual of one
             refinement iteration
  sweep      mgp_rbgs_sweep_*: one Gauss-Seidel sweep
  jacobi     mgp_bc_neumann_faces_* and mgp_jacobi_*: one Jacobi sweep

Face strings are 'D' / 'N' per face in the order north, south, east, west,
top, bottom (y high, y low, x high, x low, z high, z low).
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "multigrid-poisson_amd"))
import mgp  # noqa: E402

KERNELS = ("pair", "correct", "descend", "update", "sweep", "jacobi")
TYPES = {"f64": torch.float64, "f32": torch.float32}


def listed():
    return [
        # the reference's documented 65^3 size (4 levels, 2 + 2 sweeps, ten
        # V-cycles in reference mode): launches and latency decide
        {"name": "vcycles 65 reference", "kind": "vcycles", "nx": 65, "ny": 65, "nz": 65, "levels": 4, "cycles": 10},
        # an everyday FP64 solve with Neumann sides, to 1e-10
        {"name": "solve f64 257", "kind": "solve", "dtype": "f64", "nx": 257, "ny": 257, "nz": 129, "levels": 5,
         "bc": "NNNNDD", "tol": 1e-10},
        # the headline solve: the largest grid, Neumann x and y faces
        {"name": "solve f64 1025", "kind": "solve", "dtype": "f64", "nx": 1025, "ny": 1025, "nz": 513, "levels": 7,
         "bc": "NNNNDD", "tol": 1e-10},
        # FP32 cycles inside FP64 refinement, all faces Dirichlet
        {"name": "solve mixed 513", "kind": "solve", "dtype": "mixed", "nx": 513, "ny": 513, "nz": 257, "levels": 6,
         "bc": "DDDDDD", "tol": 1e-10},
        # a parameter study: many small uneven problems at once
        {"name": "batch 24", "kind": "batch", "count": 24, "tol": 1e-10},
        # a serving burst of mixed shapes and face types
        {"name": "server 16", "kind": "server", "count": 16, "kmin": 5, "kmax": 8},
        # the smoother's pair of sweeps in FP32 on a ragged grid (an
        # integrator's own cycle; no 2^k + 1 sizes)
        {"name": "pair f32 ragged", "kind": "pair", "dtype": "f32", "nx": 801, "ny": 610, "nz": 417, "bc": "DNNDND"},
        # the way up on the headline's finest level
        {"name": "correct f64 1025", "kind": "correct", "dtype": "f64", "nx": 1025, "ny": 1025, "nz": 513,
         "bc": "NNNNDD"},
        # the way down on the next finer level's size
        {"name": "descend f64 513", "kind": "descend", "dtype": "f64", "nx": 513, "ny": 513, "nz": 257,
         "bc": "NNNNDD"},
        # the update + residual of one refinement iteration on the finest level
        {"name": "update mixed 1025", "kind": "update", "dtype": "f64", "nx": 1025, "ny": 1025, "nz": 513,
         "bc": "DDDDDD"},
        # one sweep on a small ragged level
        {"name": "sweep f64 small", "kind": "sweep", "dtype": "f64", "nx": 129, "ny": 150, "nz": 77, "bc": "NDDDDN"},
        # the other smoother, reference arithmetic
        {"name": "jacobi f64", "kind": "jacobi", "dtype": "f64", "mode": "reference", "nx": 385, "ny": 353, "nz": 321,
         "bc": "DDNDND"},
    ]


def draw(rng):
    kind = rng.choice(KERNELS + KERNELS + ("solve", "solve", "solve", "vcycles", "batch", "server"))
    c = {"kind": kind}
    if kind in KERNELS:
        while True:
            n = [int(round(math.exp(rng.uniform(math.log(33), math.log(1100))))) for _ in range(3)]
            if n[0] * n[1] * n[2] <= 500_000_000:
                break
        if kind in ("correct", "descend"):
            n = [v | 1 for v in n]
        c.update(nx=n[0], ny=n[1], nz=n[2], dtype="f64" if kind == "update" else rng.choice(("f64", "f32")),
                 bc=_faces(rng))
        if kind == "jacobi":
            c["mode"] = rng.choice(("reference", "consistent"))
    elif kind in ("solve", "vcycles"):
        k = rng.randint(2, 5)
        while True:
            n = [rng.randint(2, 16) * 2 ** k + 1 for _ in range(2)] + [rng.randint(2, 8) * 2 ** k + 1]
            if n[0] * n[1] * n[2] <= 150_000_000:
                break
        c.update(nx=n[0], ny=n[1], nz=n[2], levels=k + 1)
        if kind == "solve":
            c.update(dtype=rng.choice(("f64", "mixed")), bc=_faces(rng)[:4] + "DD", tol=rng.choice((1e-8, 1e-9, 1e-10)))
        else:
            c.update(cycles=rng.randint(4, 12))
    elif kind == "batch":
        c.update(count=rng.randint(4, 32), tol=rng.choice((1e-8, 1e-10)))
    else:
        c.update(count=rng.randint(4, 20), kmin=5, kmax=rng.randint(6, 8))
    return c


def _faces(rng):
    while True:
        bc = "".join(rng.choice("DN") for _ in range(6))
        if "D" in bc:
            return bc


# --------------------------------------------------------------- shared parts

def _dims(c):
    return c["nx"], c["ny"], c["nz"]


def _halo(bc):
    return tuple(1 if ch == "N" else 0 for ch in bc)  # N, S, E, W, T, B


def _box(n, bc):
    N, S, E, W, T, B = (1 if ch == "D" else 0 for ch in bc)
    return (W, n[0] - E, S, n[1] - N, B, n[2] - T)


def _inner(t, n, halo):
    N, S, E, W, T, B = halo
    return t[W:W + n[0], S:S + n[1], B:B + n[2]]


def _descriptor(t, n, halo):
    a = mgp.Array()
    a.data = t.data_ptr()
    a.shape[:] = list(n)
    a.halo[:] = list(halo)
    a.stride[:] = list(t.stride())
    return a


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _coarse(n):
    return tuple((v - 1) // 2 + 1 for v in n)


def _kernel_inputs(case, seed):
    """Random level data: u of order 1, f of order 1 / h^2 (so that both count
    in an update), the Neumann faces' data and, by kind, the coarse correction
    or the refinement's lo word and correction."""
    n, bc, dt = _dims(case), case["bc"], TYPES[case["dtype"]]
    h = 1.0 / (n[0] - 1)
    g = _gen(seed)
    make = lambda shape, scale=1.0, dtype=dt: torch.randn(shape, generator=g, device="cuda", dtype=dtype).mul_(scale)  # noqa: E731
    d = {"n": n, "bc": bc, "halo": _halo(bc), "box": _box(n, bc), "h": h,
         "u": make(n), "f": make(n, 1.0 / (h * h))}
    face = {0: (n[0], n[2]), 1: (n[0], n[2]), 2: (n[1], n[2]), 3: (n[1], n[2]), 4: (n[0], n[1]), 5: (n[0], n[1])}
    d["g"] = {q: make(face[q], 0.1 / h) for q in range(6) if bc[q] == "N"}
    if case["kind"] == "correct":
        d["c"] = make(_coarse(n), 0.1)
    if case["kind"] == "update":
        d["lo"] = make(n, 1e-17, torch.float32)
        d["e"] = make(n, 1e-4, torch.float32)
    return d


def _modes(case, seed, count=4):
    """Random smooth right-hand sides as eigenmodes of the discrete operator:
    per axis (kind of mode by its two faces, wave number), and an amplitude."""
    r = np.random.default_rng(seed)
    N, S, E, W, T, B = case.get("bc", "DDDDDD")
    out = []
    for _ in range(count):
        k = r.integers(1, 6, size=3)
        out.append(([(W + E, int(k[0])), (S + N, int(k[1])), (B + T, int(k[2]))], float(r.normal())))
    return out


def _mode_axis(spec, n):
    """(values at the n points, 4 sin^2(theta / 2)) of one axis of a mode."""
    kind, m = spec
    m = {"DD": m, "NN": m, "DN": m + 0.5, "ND": m + 0.5}[kind]
    theta = math.pi * m / (n - 1)
    x = np.arange(n) * theta
    v = np.sin(x) if kind[0] == "D" else np.cos(x)
    if kind[0] == "D":
        v[0] = 0.0
    if kind[1] == "D":
        v[-1] = 0.0
    return v, 4.0 * math.sin(theta / 2) ** 2


def _mode_field(modes, n, h, solution, out=None):
    """f (or, with solution, the discrete solution of L u = f) on the grid."""
    out = torch.zeros(n, dtype=torch.float64, device="cuda") if out is None else out.zero_()
    for axes, amp in modes:
        v, lam = zip(*[_mode_axis(a, m) for a, m in zip(axes, n)])
        if solution:
            amp = -amp * h * h / sum(lam)
        x, y, z = (torch.as_tensor(a, device="cuda") for a in v)
        out.add_(torch.outer(x, y)[:, :, None] * z[None, None, :], alpha=amp)
    return out


class _Memory:
    """Device memory of the framework seen by torch (no copy).  A tensor made
    of it holds this object, and so the solver that owns the memory."""

    def __init__(self, a, owner):
        self.owner = owner
        self.p = (a.shape[0] + a.halo[2] + a.halo[3], a.shape[1] + a.halo[0] + a.halo[1],
                  a.shape[2] + a.halo[4] + a.halo[5])
        self.__cuda_array_interface__ = {"shape": self.p, "typestr": "<f8", "data": (a.data, False), "version": 2}


def _view(solver, which):
    """A solver array's shape (halos dropped) as a tensor on its own memory."""
    a = solver.device_array(which)
    t = torch.as_tensor(_Memory(a, solver), device="cuda")
    v = _inner(t, tuple(a.shape), tuple(a.halo))
    v.owner = solver
    return v


def _requests(case, seed):
    """Requests of 2^k + 1 points per axis, face types per face, four sine
    modes each that vanish on every face of the box."""
    shapes = np.random.default_rng(case["count"])  # the shapes of a burst stay, its data change
    r = np.random.default_rng(seed)
    out = []
    while len(out) < case["count"]:
        n = [int(2 ** k) for k in shapes.integers(case["kmin"], case["kmax"] + 1, size=3)]
        bc = "".join("N" if v else "D" for v in shapes.integers(0, 2, size=6))
        if len(out) % 2:
            bc = "DDDDDD"
        modes = []
        for _ in range(4):
            k = r.integers(1, 5, size=3)
            modes.append(tuple(int(k[a]) * max(1, n[0] // n[a]) for a in range(3)) + (float(r.normal()),))
        if "D" in bc:
            out.append((tuple(v + 1 for v in n), bc, modes))
    return out


def _batch_problems(case, seed):
    shapes = np.random.default_rng(case["count"])  # the shapes of a study stay, its data change
    r = np.random.default_rng(seed)
    out = []
    for _ in range(case["count"]):
        n = tuple(int(v) for v in shapes.choice([33, 65, 129], size=3))
        out.append((n, [([("DD", int(k)) for k in r.integers(1, 9, size=3)], float(r.normal())) for _ in range(4)]))
    return out


# ------------------------------------------------------------------- prepare

def prepare(case, seed):
    kind = case["kind"]
    if kind in KERNELS:
        return _prepare_kernel(case, seed)
    if kind == "batch":
        problems = _batch_problems(case, seed)
        b = mgp.Batch([n for n, _ in problems], relaxation=mgp.JACOBI, nsmooth=3, omega=6.0 / 7.0, maxiter=60,
                      tolerance=case["tol"])
        for p, (n, modes) in enumerate(problems):
            b.set_rhs(p, _mode_field(modes, n, 1.0 / (n[0] - 1), False).cpu().numpy())
        return {"case": case, "batch": b}
    if kind == "server":
        s = mgp.Server(hbm_budget=8 << 30, max_active=8, tolerance=1e-8)
        return {"case": case, "server": s, "requests": _requests(case, seed)}
    n = _dims(case)
    h = 1.0 / (n[0] - 1)
    if kind == "vcycles":
        s = mgp.Solver(n, case["levels"], h, bc="DDDDDD", mode=mgp.REFERENCE, relaxation=mgp.GAUSS_SEIDEL,
                       restriction=mgp.FULL_WEIGHTING, problem=None, maxiter=case["cycles"], tolerance=0.0)
    else:
        s = mgp.Solver(n, case["levels"], h, bc=case["bc"], mode=mgp.CONSISTENT, relaxation=mgp.GAUSS_SEIDEL,
                       restriction=mgp.FULL_WEIGHTING, problem=None,
                       dtype=mgp.F64 if case["dtype"] == "f64" else mgp.MIXED, maxiter=40, tolerance=case["tol"],
                       coarse_sweeps=32)
    mgp.call("mgp_solver_to_device_zero", s.h)
    _mode_field(_modes(case, seed), n, h, False, out=_view(s, "f"))
    torch.cuda.synchronize()
    return {"case": case, "solver": s}


def _prepare_kernel(case, seed):
    d = _kernel_inputs(case, seed)
    n, halo, kind = d["n"], d["halo"], case["kind"]
    N, S, E, W, T, B = halo
    pshape = (n[0] + E + W, n[1] + N + S, n[2] + T + B)
    s = {"case": case, "t": {}, "a": {}, "keep": d["g"]}

    def array(name, src=None, dtype=None):
        t = torch.zeros(pshape, dtype=dtype or d["u"].dtype, device="cuda")
        if src is not None:
            _inner(t, n, halo).copy_(src)
        s["t"][name] = t
        s["a"][name] = _descriptor(t, n, halo)

    array("u", d["u"])
    array("f", d["f"])
    if kind == "descend":
        array("r")
        s["t"]["c"] = torch.zeros(_coarse(n), dtype=d["u"].dtype, device="cuda")
        s["a"]["c"] = _descriptor(s["t"]["c"], _coarse(n), (0,) * 6)
    elif kind == "update":
        array("r")
        array("out")
        array("lo", d["lo"], torch.float32)
        array("e", d["e"], torch.float32)
        array("lo_new", None, torch.float32)
        array("f32", None, torch.float32)
        s["norm"] = torch.zeros(1, dtype=torch.float64, device="cuda")
    else:
        array("out")
    if kind == "correct":
        s["t"]["c"] = d["c"]
        s["a"]["c"] = _descriptor(d["c"], _coarse(n), (0,) * 6)
    F = mgp.Faces()
    for q in range(6):
        F.type[q] = mgp.NEUMANN if q in d["g"] else mgp.DIRICHLET
        F.g[q] = d["g"][q].data_ptr() if q in d["g"] else None
    F.h = d["h"]
    s.update(F=F, box=(ctypes.c_int64 * 6)(*d["box"]), h=d["h"], n=n, halo=halo)
    torch.cuda.synchronize()
    return s


# ----------------------------------------------------------------------- run

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind in KERNELS:
        return _run_kernel(s, case, kind)
    if kind == "batch":
        b = s["batch"]
        b.solve()
        stats = [b.stats(p) for p in range(case["count"])]
        return {"u": [b.solution(p) for p in range(case["count"])], "iterations": np.array([i for i, _ in stats])}
    if kind == "server":
        ids = [s["server"].submit(*r) for r in s["requests"]]
        got = [s["server"].wait(i) for i in ids]
        return {"u": [u for _, u in got], "iterations": np.array([r.iterations for r, _ in got]),
                "status": np.array([r.status for r, _ in got])}
    solver = s["solver"]
    solver.reset()
    if kind == "vcycles":
        it, rr, _ = solver.solve("Vcycle", 2, 1.0)
    else:
        it, rr, _ = solver.solve("Fcycle", 2, 1.0)
    return {"u": _view(solver, "u"), "iterations": it, "rel_res": rr}


def _run_kernel(s, case, kind):
    ref = {k: ctypes.byref(a) for k, a in s["a"].items()}
    F, box, x = ctypes.byref(s["F"]), ctypes.byref(s["box"]), case["dtype"]
    out = lambda name: _inner(s["t"][name], s["n"], s["halo"])  # noqa: E731
    if kind == "descend":
        mgp.call("mgp_bc_neumann_faces_" + x, ref["u"], F, None)
        mgp.call("mgp_residual_restrict_fw_" + x, mgp.CONSISTENT, ref["u"], ref["f"], ref["r"], ref["c"], box, s["h"],
                 None)
        return s["t"]["c"]
    if kind == "update":
        norm = s["norm"].data_ptr()
        mgp.call("mgp_zero_scalars", norm, 1, None)
        mgp.call("mgp_update_residual_hilo_f64_f32", ref["u"], ref["out"], ref["lo"], ref["lo_new"], ref["e"], ref["f"],
                 ref["r"], ref["f32"], F, box, norm, None)
        return {"u": out("out"), "lo": out("lo_new"), "r": out("f32"), "norm": s["norm"]}
    if kind == "jacobi":
        mode = mgp.REFERENCE if case["mode"] == "reference" else mgp.CONSISTENT
        mgp.call("mgp_bc_neumann_faces_" + x, ref["u"], F, None)
        mgp.call("mgp_jacobi_" + x, mode, ref["out"], ref["u"], ref["f"], box, 6.0 / 7.0, s["h"], None)
        return out("out")
    args = (mgp.CONSISTENT, ref["u"], ref["out"], ref["f"], F, box, 1.0)
    if kind == "sweep":
        mgp.call("mgp_rbgs_sweep_" + x, *args, None)
    elif kind == "pair":
        mgp.call("mgp_rbgs_sweep2_" + x, *args, None)
    else:
        mgp.call("mgp_rbgs_sweep2_prolong_" + x, *args, ref["c"], None)
    return out("out")


# ---------------------------------------------------------------------- work

def work(case):
    """Bytes: inputs read once and outputs written once.  Flops: the stencil
    operations of the call; for whole solves those of the fewest cycles that
    can reach the tolerance at one decade per cycle."""
    kind = case["kind"]
    if kind == "batch":
        pts = sum(n[0] * n[1] * n[2] for n, _ in _batch_problems(case, 0))
        return {"bytes": 24.0 * pts, "flops": 90.0 * pts * -math.log10(case["tol"])}
    if kind == "server":
        pts = sum(n[0] * n[1] * n[2] for n, _, _ in _requests(case, 0))
        return {"bytes": 8.0 * pts, "flops": 90.0 * pts * 8}
    n = _dims(case)
    pts = float(n[0] * n[1] * n[2])
    if kind == "vcycles":
        return {"bytes": 24.0 * pts, "flops": 90.0 * pts * case["cycles"]}
    if kind == "solve":
        return {"bytes": 24.0 * pts, "flops": 90.0 * pts * -math.log10(case["tol"])}
    w = 8.0 if case["dtype"] == "f64" else 4.0
    if kind == "update":
        return {"bytes": 40.0 * pts, "flops": 40.0 * pts}
    if kind == "descend":
        return {"bytes": 2.125 * w * pts, "flops": 22.0 * pts}
    sweeps = 2 if kind in ("pair", "correct") else 1
    extra = 0.125 if kind == "correct" else 0.0
    return {"bytes": (3 + extra) * w * pts, "flops": 13.0 * sweeps * pts}


# --------------------------------------------------------------------- exact

def exact(case, seed):
    kind = case["kind"]
    if kind in KERNELS:
        return _exact_kernel(case, seed)
    if kind == "batch":
        u = [_mode_field(m, n, 1.0 / (n[0] - 1), True).cpu().numpy() for n, m in _batch_problems(case, seed)]
        return {"u": u, "iterations": None}
    if kind == "server":
        u = []
        for n, bc, modes in _requests(case, seed):
            if bc != "DDDDDD":
                u.append(None)
                continue
            h = 1.0 / (n[0] - 1)
            u.append(_mode_field([([("DD", k * (m - 1) // (n[0] - 1)) for k, m in zip(w[:3], n)], w[3])
                                  for w in modes], n, h, True).cpu().numpy())
        return {"u": u, "iterations": None, "status": None}
    n = _dims(case)
    return {"u": _mode_field(_modes(case, seed), n, 1.0 / (n[0] - 1), True), "iterations": None, "rel_res": None}


def _padded(x, n):
    p = torch.zeros([v + 2 for v in n], dtype=torch.float64, device="cuda")
    p[1:-1, 1:-1, 1:-1] = x
    return p


def _ghosts(p, d):
    two_h, n = 2.0 * d["h"], d["n"]
    i, o = slice(1, -1), {q: g.double() for q, g in d["g"].items()}
    if 0 in o:
        p[i, n[1] + 1, i] = two_h * o[0] + p[i, n[1] - 1, i]
    if 1 in o:
        p[i, 0, i] = -two_h * o[1] + p[i, 2, i]
    if 2 in o:
        p[n[0] + 1, i, i] = two_h * o[2] + p[n[0] - 1, i, i]
    if 3 in o:
        p[0, i, i] = -two_h * o[3] + p[2, i, i]
    if 4 in o:
        p[i, i, n[2] + 1] = two_h * o[4] + p[i, i, n[2] - 1]
    if 5 in o:
        p[i, i, 0] = -two_h * o[5] + p[i, i, 2]


def _neighbours(p, b):
    """Sum of u_nb - u over the box (b in shape indices, p padded by one)."""
    x, y, z = (slice(b[2 * a] + 1, b[2 * a + 1] + 1) for a in range(3))
    up = lambda s: slice(s.start + 1, s.stop + 1)  # noqa: E731
    dn = lambda s: slice(s.start - 1, s.stop - 1)  # noqa: E731
    c = p[x, y, z]
    s = (p[up(x), y, z] - c).add_(p[dn(x), y, z] - c)
    s.add_(p[x, up(y), z] - c).add_(p[x, dn(y), z] - c)
    return s.add_(p[x, y, up(z)] - c).add_(p[x, y, dn(z)] - c)


def _sweep(p, d, omega):
    b = d["box"]
    x, y, z = (slice(b[2 * a] + 1, b[2 * a + 1] + 1) for a in range(3))
    f = d["f"][b[0]:b[1], b[2]:b[3], b[4]:b[5]]
    par = [torch.arange(b[2 * a], b[2 * a + 1], device="cuda") for a in range(3)]
    red = (par[0][:, None, None] + par[1][None, :, None] + par[2][None, None, :]) % 2 == 0
    for colour in (red, ~red):
        _ghosts(p, d)
        s = _neighbours(p, b).sub_(f.double(), alpha=d["h"] ** 2)
        p[x, y, z] += torch.where(colour, s, 0.0).mul_(omega / 6.0)


def _interpolate(c, axis):
    shape = list(c.shape)
    shape[axis] = 2 * shape[axis] - 1
    out = torch.empty(shape, dtype=torch.float64, device=c.device)
    o, m = out.movedim(axis, 0), c.movedim(axis, 0)
    o[0::2] = m
    o[1::2] = 0.5 * (m[:-1] + m[1:])
    return out


def _weight(r, axis):
    m = r.movedim(axis, 0)
    m = torch.cat([m[:1], m, m[-1:]])
    return (0.25 * m[0:-2:2] + 0.5 * m[1:-1:2] + 0.25 * m[2::2]).movedim(0, axis)


def _exact_kernel(case, seed):
    d = _kernel_inputs(case, seed)
    n, b, kind, h = d["n"], d["box"], case["kind"], d["h"]
    inside = tuple(slice(b[2 * a], b[2 * a + 1]) for a in range(3))
    u = d["u"].double()
    if kind == "correct":
        c = d["c"].double()
        for a in range(3):
            c = _interpolate(c, a)
        u = u + c
    if kind == "update":
        t = d["e"].double() + d["lo"].double()
        hi = u + t
        bb = hi - u
        lo = (u - (hi - bb)) + (t - bb)
        p, q = _padded(hi, n), _padded(lo, n)
        _ghosts(p, d)
        _ghosts(q, dict(d, g={k: torch.zeros_like(g) for k, g in d["g"].items()}))
        s = _neighbours(p, b).add_(_neighbours(q, b))
        r = torch.zeros(n, dtype=torch.float64, device="cuda")
        r[inside] = d["f"][inside].double() - s / (h * h)
        return {"u": hi, "lo": lo, "r": r, "norm": r.abs().max().reshape(1)}
    p = _padded(u, n)
    del u
    if kind in ("sweep", "pair", "correct"):
        for _ in range(1 if kind == "sweep" else 2):
            _sweep(p, d, 1.0)
        return p[1:-1, 1:-1, 1:-1]
    _ghosts(p, d)
    s = _neighbours(p, b)
    out = torch.zeros(n, dtype=torch.float64, device="cuda")
    if kind == "jacobi":
        x, y, z = (slice(b[2 * a] + 1, b[2 * a + 1] + 1) for a in range(3))
        out[inside] = p[x, y, z] + (6.0 / 7.0 / 6.0) * (s - h * h * d["f"][inside].double())
        return out
    out[inside] = d["f"][inside].double() - s / (h * h)
    for a in range(3):
        out = _weight(out, a)
    return out
