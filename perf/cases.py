"""The workloads whose speed this framework is judged by: whole uses of its
solver, as a program makes them, with the outputs such a program takes.

Each case is one of these uses ("kind"):

  frame     a running simulation is advanced to its next frame and its state
            taken out (the vortex and Taylor-Green runs of bench.py)
  solve     one problem from its initial state to an end time
            (advection pulse, cavity, dam break, Sod tube)
  loop      the driver loop: run_ssprk3_loop with diagnostics rows
  adaptive  dt from the device CFL reduction before every step
  ensemble  a Batch of instances of different size, advanced to a frame

in one arithmetic form ("f64": plain FP64, "f32": FP32-MFMA, whose outputs
are kept in that precision).  Meshes are triangles (two
per square) or tetrahedra (six per cube).

exact() computes the same outputs with an independent FP64 discontinuous
Galerkin method in torch: exact rational reference operators, the lattice's
own connectivity, and the textbook fluxes.
"""
import functools
import itertools
import math
from fractions import Fraction

import numpy as np
import torch

import mojoxm_amd as M

GAMMA = 1.4


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # The smallest meshes: every stage is a handful of tiles, so launches
        # and the dependent chain of one tile are what a step costs.  The
        # driver loop steps one step per call and writes a row per frame.
        dict(name="alfven_16_loop_f32", kind="loop", problem="alfven", nx=16, ny=16, P=3, form="f32", steps=200),
        # A small ragged mesh whose time step follows the measured wave speed.
        dict(name="vortex_33_adaptive_f64", kind="adaptive", problem="vortex", nx=33, ny=33, P=2, form="f64", steps=48),
        # The Gaussian pulse through the unit cube and back (one component).
        dict(name="advection_16_f64", kind="solve", problem="advection", nx=16, ny=16, nz=16, P=2, form="f64",
             steps=462),
        # Requests of the serving stream: a limited dam break and a limited
        # Sod tube between walls, and a P = 4 cavity between conducting ones.
        dict(name="dam_break_75_p2_f64", kind="solve", problem="dam_break", nx=75, ny=75, P=2, form="f64", steps=300),
        dict(name="cavity_113_p4_f32", kind="solve", problem="cavity", nx=113, ny=113, P=4, form="f32", steps=400),
        dict(name="sod_192_f64", kind="solve", problem="sod", nx=192, ny=192, P=3, form="f64", steps=400),
        # The headline vortex, a quarter of its run per frame, in both forms,
        # and the same problem on a mesh whose state exceeds the caches.
        dict(name="vortex_128_f32", kind="frame", problem="vortex", nx=128, ny=128, P=3, form="f32", steps=1000),
        dict(name="vortex_128_f64", kind="frame", problem="vortex", nx=128, ny=128, P=3, form="f64", steps=1000),
        dict(name="vortex_512_f32", kind="frame", problem="vortex", nx=512, ny=512, P=3, form="f32", steps=400),
        # Taylor-Green with its kinetic energy and enstrophy per frame: an
        # odd mid-sized mesh in FP32 and the full one in FP64.
        dict(name="tgv_19_f32", kind="frame", problem="tgv", nx=19, ny=19, nz=19, P=3, form="f32", steps=200),
        dict(name="tgv_32_f64", kind="frame", problem="tgv", nx=32, ny=32, nz=32, P=3, form="f64", steps=200),
        # The batched ensemble: Alfven waves on meshes of 16..96 squares.
        dict(name="ensemble_24_f32", kind="ensemble", problem="alfven", count=24, n_min=16, n_max=96, P=3, form="f32",
             steps=400),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    form = rng.choice(["f32", "f64"])
    problem = rng.choice(["vortex", "vortex", "tgv", "advection", "alfven", "dam_break", "sod", "cavity", "ensemble"])
    if problem == "ensemble":
        return dict(kind="ensemble", problem="alfven", count=rng.randint(4, 20), n_min=16, n_max=log(32, 96), P=3,
                    form=form, steps=rng.randint(100, 300))
    case = dict(problem=problem, form=form)
    if problem in ("tgv", "advection"):
        n = log(6, 26)
        case.update(nx=n, ny=max(4, int(n * rng.uniform(0.7, 1.2))), nz=max(4, int(n * rng.uniform(0.7, 1.2))),
                    P=rng.choice([2, 3]))
    else:
        n = log(16, 400 if problem == "vortex" else 224)
        case.update(nx=n, ny=max(8, int(n * rng.uniform(0.6, 1.2))), P=rng.choice([2, 3, 3, 4]))
    if problem == "sod":  # the limiter bounds the density only: P = 4 tubes leave the physical states
        case["P"] = min(case["P"], 3)
    if problem == "dam_break":
        case["P"] = 2
    if problem == "alfven":
        case["kind"] = rng.choice(["loop", "frame"])
    elif problem == "vortex":
        case["kind"] = rng.choice(["frame", "frame", "adaptive"])
    else:
        case["kind"] = "frame" if problem == "tgv" else "solve"
    # about a tenth of a second at most
    per_step = 20e-6 + 1.2e-11 * 3 * values(case)
    case["steps"] = min(rng.randint(100, 600), int(0.1 / per_step))
    if case["kind"] == "adaptive":
        case["steps"] = min(case["steps"], 64)
    return case


# ---------------------------------------------------------------------------
# sizes
# ---------------------------------------------------------------------------
NC = dict(vortex=5, tgv=5, advection=1, alfven=7, dam_break=3, sod=5, cavity=6)
LIMITED = ("dam_break", "sod")
# flops of one nodal flux, one numerical flux and one node's stage combine
FLUX = dict(vortex=(25, 150, 35), tgv=(40, 110, 35), advection=(3, 8, 5), alfven=(70, 190, 35), dam_break=(20, 60, 15),
            sod=(25, 150, 35), cavity=(15, 40, 35))


def dims(case):
    return 3 if "nz" in case else 2


def nodes(nd, P):
    return (P + 1) * (P + 2) * (P + 3) // 6 if nd == 3 else (P + 1) * (P + 2) // 2


def elements(case):
    return 6 * case["nx"] * case["ny"] * case["nz"] if "nz" in case else 2 * case["nx"] * case["ny"]


def values(case):
    return elements(case) * nodes(dims(case), case["P"]) * NC[case["problem"]]


def work(case):
    """Three stages per step, each reading its input (and the combine's first
    operand, where that is another state) and writing its output: 8 states
    per step; plus the state handed over.  The operations are the
    contractions, one flux per node, one numerical flux per face node."""
    if case["kind"] == "ensemble":
        parts = [work(dict(case, kind="frame", nx=n, ny=n)) for n in _ensemble_sizes(case)]
        return {k: float(sum(p[k] for p in parts)) for k in ("bytes", "flops")}
    nd, P, nc = dims(case), case["P"], NC[case["problem"]]
    K, n, nfp, nf = elements(case), nodes(nd, P), nodes(nd - 1, P) if nd == 3 else P + 1, nd + 1
    word = 8 if case["form"] == "f64" else 4
    nodal, face, combine = FLUX[case["problem"]]
    per = 2 * n * (nd * n + nf * nfp) * nc + n * (nodal + combine + 2 * nd * nd * nc) + nf * nfp * face / 2
    moved = 8 * K * n * nc * word * case["steps"]
    if case["kind"] == "adaptive":
        moved += K * n * nc * word * case["steps"]
    return {"bytes": float(moved + K * n * nc * 8 * (2 if case["kind"] == "solve" else 1)),
            "flops": float(3 * case["steps"] * K * per)}


# ---------------------------------------------------------------------------
# problems: parameters and initial states from the seed
# ---------------------------------------------------------------------------
def _labels(nd, P):
    """Barycentric labels of the nodes: vertices, edges, faces, interior."""
    nv = nd + 1
    unit = [tuple(P if v == w else 0 for v in range(nv)) for w in range(nv)]
    edges = [(0, 1), (1, 2), (2, 0), (0, 3), (1, 3), (2, 3)][:6 if nd == 3 else 3]

    def put(**at):
        return tuple(at.get("v%d" % v, 0) for v in range(nv))

    out = list(unit)
    for a, b in edges:
        out += [put(**{"v%d" % a: P - k, "v%d" % b: k}) for k in range(1, P)]
    faces = [[v for v in range(4) if v != f] for f in range(4)] if nd == 3 else [[0, 1, 2]]
    for x, y, z in faces:
        out += [put(**{"v%d" % x: i, "v%d" % y: j, "v%d" % z: P - i - j})
                for i in range(P - 2, 0, -1) for j in range(P - i - 1, 0, -1)]
    if nd == 3:
        out += [(i, j, k, P - i - j - k) for i in range(P - 2, 0, -1) for j in range(P - i - 1, 0, -1)
                for k in range(P - i - j - 1, 0, -1)]
    return out


# corners of each element of a cell: the /-split square, the Kuhn cube
CELL = {2: [[(0, 0), (1, 0), (1, 1)], [(0, 0), (1, 1), (0, 1)]],
        3: [[tuple(c >> d & 1 for d in range(3)) for c in t] for t in
            [(0, 1, 3, 7), (0, 3, 2, 7), (0, 2, 6, 7), (0, 6, 4, 7), (0, 4, 5, 7), (0, 5, 1, 7)]]}


def _shape(case):
    return (case["nx"], case["ny"]) + ((case["nz"],) if "nz" in case else ())


def _coordinates(n, L, P):
    """Node coordinates [K, NP, ND], cells x-fastest, then the cell's elements."""
    nd = len(n)
    bary = np.array(_labels(nd, P), dtype=np.int64)
    local = np.stack([bary @ np.array(t, dtype=np.int64) for t in CELL[nd]])  # [T, NP, ND]
    cells = np.stack(np.meshgrid(*[np.arange(k) for k in n[::-1]], indexing="ij")[::-1], axis=-1).reshape(-1, 1, 1, nd)
    x = (P * cells + local[None]).astype(np.float64) * (np.array(L) / np.array(n)) / P
    return x.reshape(-1, bary.shape[0], nd)


def _problem(case, seed):
    """The physics record, box, boundaries, time step and initial state."""
    r = np.random.default_rng(seed)
    kind, P, n = case["problem"], case["P"], _shape(case)
    nd = len(n)
    L, bcs, prm = (1.0,) * nd, (0, 0) * nd, {}
    if kind == "vortex":
        L, beta = (10.0, 10.0), r.uniform(4.0, 5.0)
        c = r.uniform(3.0, 7.0, 2)
        prm = dict(gamma=GAMMA, flux="hllec")
        phys = M.physics.Euler(gamma=GAMMA, flux_type=M.physics.FLUX_HLLEC)
        speed, cfl = math.sqrt(2.0) + math.sqrt(GAMMA) + beta / (2 * math.pi), 0.15

        def ic(x):
            dx, dy = ((x[..., d] - c[d] + 5.0) % 10.0 - 5.0 for d in range(2))
            r2 = dx * dx + dy * dy
            T = 1.0 - (GAMMA - 1) * beta ** 2 / (8 * GAMMA * math.pi ** 2) * np.exp(1 - r2)
            e = beta / (2 * math.pi) * np.exp(0.5 * (1 - r2))
            rho, u, v = T ** (1 / (GAMMA - 1)), 1 - e * dy, 1 + e * dx
            return [rho, rho * u, rho * v, 0 * rho, rho * T / (GAMMA - 1) + 0.5 * rho * (u * u + v * v)]
    elif kind == "tgv":
        L, mach, s = (2 * math.pi,) * 3, 0.3, r.uniform(0, 2 * math.pi, 3)
        prm = dict(gamma=GAMMA, flux="rusanov")
        phys = M.physics.Euler(gamma=GAMMA, flux_type=M.physics.FLUX_RUSANOV)
        speed, cfl = 1 + 1 / mach, 0.2

        def ic(x):
            x, y, z = (x[..., d] + s[d] for d in range(3))
            u, v = np.sin(x) * np.cos(y) * np.cos(z), -np.cos(x) * np.sin(y) * np.cos(z)
            p = 1 / (GAMMA * mach ** 2) + (np.cos(2 * x) + np.cos(2 * y)) * (np.cos(2 * z) + 2) / 16
            return [1 + 0 * u, u, v, 0 * u, p / (GAMMA - 1) + 0.5 * (u * u + v * v)]
    elif kind == "advection":
        c, sigma = r.uniform(0.3, 0.7, 3), r.uniform(0.09, 0.12)
        prm = dict(v=(1.0, 1.0, 1.0))
        phys = M.physics.Advection(1.0, 1.0, 1.0)
        speed, cfl = math.sqrt(3.0), 0.3

        def ic(x):
            d = (x - c + 0.5) % 1.0 - 0.5
            return [np.exp(-(d * d).sum(-1) / (2 * sigma * sigma))]
    elif kind == "alfven":
        a, b = [(1, 0), (3, 1), (2, 1), (3, 2), (1, 1), (2, 3), (1, 2), (1, 3)][r.integers(8)]
        amp, kn, ph, g = r.uniform(0.01, 0.2), math.hypot(a, b), r.uniform(0, 1), 5 / 3
        ch = amp + math.sqrt(g * 0.1 + 1 + amp * amp)
        prm = dict(gamma=g, ch=ch, alpha=ch / 0.18)
        phys = M.physics.MHDGLM2D(gamma=g, c_h=ch, alpha_d=ch / 0.18)
        speed, cfl = ch, 0.15

        def ic(x):
            s = amp * np.sin(2 * math.pi * (a * x[..., 0] + b * x[..., 1] + ph))
            u, v = -s * b / kn, s * a / kn
            Bx, By = (a + s * b) / kn, (b - s * a) / kn
            return [1 + 0 * s, u, v, Bx, By, 0.1 / (g - 1) + 0.5 * (u * u + v * v + Bx * Bx + By * By), 0 * s]
    elif kind == "dam_break":
        ratio, bcs = r.uniform(2.0, 10.0), (1, 1, 1, 1)
        prm = dict(g=9.81)
        phys = M.physics.ShallowWater2D(g=9.81, hll=True)
        speed, cfl = math.sqrt(9.81 * ratio), 0.2

        def ic(x):
            h = np.where(x[..., 0] < 0.5, ratio, 1.0)
            return [h, 0 * h, 0 * h]
    elif kind == "sod":
        bcs, m = (2, 2, 1, 1), r.uniform(0.45, 0.55)
        prm = dict(gamma=GAMMA, flux="hlle")
        phys = M.physics.Euler(gamma=GAMMA, flux_type=M.physics.FLUX_HLLE)
        speed, cfl = 2 * math.sqrt(GAMMA), 0.15

        def ic(x):
            s = 0.5 * (np.tanh((x[..., 0] - m) * n[0] / 8) + 1)
            rho = 1 - 0.875 * s
            return [rho, 0 * s, 0 * s, 0 * s, (1 - 0.9 * s) / (GAMMA - 1)]
    else:  # cavity
        (k, l), bcs, z = r.integers(1, 5, 2), (1, 1, 1, 1), r.uniform(0.5, 1.5)
        prm = dict(c=1.0)
        phys = M.physics.Maxwell2D(c=1.0)
        speed, cfl = 1.0, 0.2

        def ic(x):
            e = z * np.sin(k * math.pi * x[..., 0]) * np.sin(l * math.pi * x[..., 1])
            return [0 * e, 0 * e, e, 0 * e, 0 * e, 0 * e]
    h = min(Ld / nd_ for Ld, nd_ in zip(L, n))
    q0 = np.stack(ic(_coordinates(n, L, P)), axis=-1)
    if case["form"] == "f32":  # states the form can hold
        q0 = q0.astype(np.float32).astype(np.float64)
    return dict(case=case, n=n, L=L, bcs=bcs, prm=prm, phys=phys, dt=cfl * h / (speed * (2 * P + 1)), q0=q0, h=h)


def _ensemble_sizes(case):
    r = np.random.default_rng(case["count"])
    lo, hi = case["n_min"], case["n_max"]
    return [int(round(lo * (hi / lo) ** u)) for u in r.uniform(0, 1, case["count"])]


def _ensemble(case, seed):
    return [_problem(dict(case, nx=n, ny=n), [seed, i]) for i, n in enumerate(_ensemble_sizes(case))]


# ---------------------------------------------------------------------------
# a program's set-up, and one pass
# ---------------------------------------------------------------------------
def _form(case):
    return M.PREC_FP64 if case["form"] == "f64" else M.PREC_FP32_MFMA


def prepare(case, seed):
    if case["kind"] == "ensemble":
        b = M.batch.Batch(_form(case))
        ids = [b.add(p["n"], p["L"], p["phys"], case["P"], p["q0"], p["dt"], 1 << 30) for p in _ensemble(case, seed)]
        return dict(case=case, batch=b, ids=ids)
    p = _problem(case, seed)
    bcs = (M.BoundaryConditions if dims(case) == 3 else M.BoundaryConditions2D)(*p["bcs"])
    s = M.Solver(p["n"], p["L"], p["phys"], P=case["P"], bcs=bcs, precision=_form(case))
    if case["problem"] in LIMITED:
        s.enable_cell_limiter(True, 0.1)
    s.set_state(p["q0"])
    s.autotune(p["dt"], 5)
    if case["kind"] in ("frame", "solve"):
        s.prepare_steps(p["dt"], case["steps"])
    return dict(case=case, solver=s, dt=p["dt"], h=p["h"], q0=p["q0"])


def _state(case, q):
    return q if case["form"] == "f64" else q.astype(np.float32)


def _row(case, d):
    return {k: _state(case, getattr(d, k)) for k in ("integral", "squared", "maxabs")}


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "ensemble":
        b = state["batch"]
        b.step(case["steps"])
        return [_state(case, b.get_state(i)) for i in state["ids"]]
    s, dt, steps = state["solver"], state["dt"], case["steps"]
    if kind == "loop":
        rows = []
        s.set_state(state["q0"])
        M.run_ssprk3_loop(s, dt, (steps - 0.5) * dt, num_frames=4,
                          on_frame=lambda sv, t: rows.append(_row(case, sv.diagnostics())))
        return dict(rows=rows, q=_state(case, s.get_state()))
    if kind == "adaptive":
        s.set_state(state["q0"])
        times = []
        for _ in range(steps):
            times.append(M.cfl_dt(s, 0.15, state["h"]))
            s.step_ssprk3(times[-1])
        return dict(dt=_state(case, np.array(times)), q=_state(case, s.get_state()))
    if kind == "solve":
        s.set_state(state["q0"])
    s.step_ssprk3(dt, steps)
    if case["problem"] == "tgv":
        d = s.diagnostics()
        return dict(energies=_state(case, np.array([d.kinetic_energy, d.enstrophy])), q=_state(case, s.get_state()))
    return _state(case, s.get_state())


# ---------------------------------------------------------------------------
# the same outputs from an independent FP64 method
# ---------------------------------------------------------------------------
def _solve_fractions(A, B):
    """A^-1 B in rational arithmetic."""
    n = len(A)
    rows = [list(a) + list(b) for a, b in zip(A, B)]
    for k in range(n):
        p = next(r for r in range(k, n) if rows[r][k])
        rows[k], rows[p] = rows[p], rows[k]
        inv = 1 / rows[k][k]
        rows[k] = [v * inv for v in rows[k]]
        for r in range(n):
            f = rows[r][k]
            if r != k and f:
                rows[r] = [a - f * b if b else a for a, b in zip(rows[r], rows[k])]
    return [r[n:] for r in rows]


def _integral(e):
    """Of the monomial with exponents e over the unit simplex."""
    return Fraction(math.prod(math.factorial(k) for k in e), math.factorial(sum(e) + len(e)))


def _monomials(nd, P):
    return [e for e in itertools.product(range(P + 1), repeat=nd) if sum(e) <= P]


def _basis(labels, P):
    """Monomials and the coefficients c[k][i] of the Lagrange basis on them."""
    nd = len(labels[0]) - 1
    mono = _monomials(nd, P)
    V = [[math.prod(Fraction(l[d + 1], P) ** e[d] for d in range(nd)) for e in mono] for l in labels]
    eye = [[Fraction(int(i == j)) for j in range(len(mono))] for i in range(len(mono))]
    return mono, _solve_fractions(V, eye)


def _mul(A, B):
    Bt = list(zip(*B))
    return [[sum(a * b for a, b in zip(r, c) if a and b) for c in Bt] for r in A]


@functools.lru_cache(maxsize=None)
def _operators(nd, P):
    """Weak derivatives D[nd][NP][NP], lift per face node [NF][NP][NFP], node
    weights, nodal derivatives and the node list of each face."""
    labels = _labels(nd, P)
    mono, c = _basis(labels, P)
    ct = [list(r) for r in zip(*c)]
    add = lambda a, b: tuple(x + y for x, y in zip(a, b))  # noqa: E731
    mass = _mul(_mul(ct, [[_integral(add(a, b)) for b in mono] for a in mono]), c)
    stiff = []
    for d in range(nd):
        low = [tuple(v - (k == d) for k, v in enumerate(e)) for e in mono]
        g = [[e[d] * _integral(add(lo, f)) if e[d] else Fraction(0) for f in mono] for e, lo in zip(mono, low)]
        stiff.append(_mul(_mul(ct, g), c))
    off = [f if nd == 3 else (f + 2) % 3 for f in range(nd + 1)]  # the vertex each face leaves out
    faces = [[i for i, l in enumerate(labels) if l[o] == 0] for o in off]
    lifted = []
    for o, fn in zip(off, faces):
        flab = [tuple(v for k, v in enumerate(labels[i]) if k != o) for i in fn]
        fm, fc = _basis(flab, P)
        G = _mul(_mul([list(r) for r in zip(*fc)], [[_integral(add(a, b)) * math.factorial(nd - 1) for b in fm] for a in fm]), fc)
        rows = [[Fraction(0)] * len(fn) for _ in labels]
        for i, g in zip(fn, G):
            rows[i] = g
        lifted.append(rows)
    right = [[v for m in stiff + lifted for v in m[i]] for i in range(len(labels))]
    sol = np.array([[float(v) for v in r] for r in _solve_fractions(mass, right)])
    NP, NFP = len(labels), len(faces[0])
    D = np.stack([sol[:, d * NP:(d + 1) * NP] for d in range(nd)])
    lift = np.stack([sol[:, nd * NP + f * NFP: nd * NP + (f + 1) * NFP] for f in range(nd + 1)])
    w = np.array([float(math.factorial(nd) * sum(ct[i][k] * _integral(e) for k, e in enumerate(mono))) for i in range(NP)])
    nodal = np.zeros((nd, NP, NP))
    for d in range(nd):
        for i, l in enumerate(labels):
            x = [Fraction(v, P) for v in l[1:]]
            dm = [e[d] * math.prod(x[k] ** (e[k] - (k == d)) for k in range(nd)) if e[d] else Fraction(0) for e in mono]
            nodal[d, i] = [float(sum(ct[j][k] * dm[k] for k in range(len(mono)))) for j in range(NP)]
    return D, lift, w, nodal, faces, off


class _Field:
    """The method on one mesh, states as [NP, NC, K] tensors."""

    def __init__(self, p):
        case = p["case"]
        self.p, self.dev = p, "cuda" if torch.cuda.is_available() else "cpu"
        n, L, P, nd = p["n"], p["L"], case["P"], len(p["n"])
        self.nd, self.P, self.NC = nd, P, NC[case["problem"]]
        D, lift, w, nodal, faces, off = _operators(nd, P)
        labels, T = _labels(nd, P), len(CELL[nd])
        cells = int(np.prod(n))
        self.K = cells * T
        put = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=self.dev)  # noqa: E731
        self.NP, self.F, self.NFP = len(labels), nd + 1, len(faces[0])
        self.D = put(np.concatenate(list(D), axis=1))                 # [NP, ND*NP]
        self.lift = put(np.concatenate(list(lift), axis=1))           # [NP, F*NFP]
        self.w, self.nodal = put(w), put(nodal)
        h = np.array(L) / np.array(n)
        corners = [np.array(t, dtype=np.int64) for t in CELL[nd]]
        J = np.stack([((c[1:] - c[0]) * h).T for c in corners])
        inv, det = np.linalg.inv(J), np.linalg.det(J)
        bary = np.array(labels, dtype=np.int64)
        at = [bary @ c for c in corners]                              # node lattice positions in the cell
        index = np.stack(np.meshgrid(*[np.arange(k) for k in n[::-1]], indexing="ij")[::-1], -1).reshape(-1, nd)
        stride = np.cumprod([1] + list(n[:-1]))
        nb_e = np.zeros((self.F, cells, T), dtype=np.int64)
        nb_n = np.zeros((self.F, self.NFP, T), dtype=np.int64)
        bc = np.zeros((self.F, cells, T), dtype=np.int64)
        normal, area = np.zeros((nd, self.F, T)), np.zeros((self.F, T))
        for t, f in itertools.product(range(T), range(self.F)):
            grad = -inv[t].sum(0) if off[f] == 0 else inv[t][off[f] - 1]
            size = np.linalg.norm(grad)
            normal[:, f, t], area[f, t] = -grad / size, det[t] * size / math.factorial(nd - 1)
            mine = [tuple(x) for x in at[t][faces[f]]]
            found = None
            for shift in itertools.product((-1, 0, 1), repeat=nd):
                for t2, f2 in itertools.product(range(T), range(self.F)):
                    theirs = {tuple(x): i for x, i in zip(at[t2][faces[f2]] + P * np.array(shift), faces[f2])}
                    if (t2, shift) != (t, (0,) * nd) and set(theirs) == set(mine):
                        found = (t2, shift, [theirs[x] for x in mine])
            t2, shift, there = found
            to = index + np.array(shift)
            nb_n[f, :, t] = there
            nb_e[f, :, t] = ((to % np.array(n)) * stride).sum(-1) * T + t2
            for d in range(nd):
                if shift[d]:
                    kind = p["bcs"][2 * d + (shift[d] > 0)]
                    if kind:
                        bc[f, (to[:, d] < 0) | (to[:, d] >= n[d]), t] = kind
        self.own = put(np.concatenate([np.array(f) for f in faces]))  # [F*NFP]
        self.nb_e = put(nb_e.reshape(self.F, self.K))
        each = lambda a: np.tile(a, cells) if a.ndim == 1 else np.tile(a, (1,) * (a.ndim - 1) + (cells,))  # noqa: E731
        self.nb_e_nodes = self.nb_e.repeat_interleave(self.NFP, 0)
        self.nb_n = put(each(nb_n.reshape(self.F * self.NFP, T)))
        self.bc = put(bc.reshape(self.F, self.K))
        self.bcs = sorted(set(np.unique(bc)) - {0})
        self.bc_nodes = self.bc.repeat_interleave(self.NFP, 0) if self.bcs else None
        self.normal = [put(each(x)).repeat_interleave(self.NFP, 0) for x in normal]
        self.scale = put(each(area / det)).repeat_interleave(self.NFP, 0)
        self.inv = [[put(each(inv[:, k, d])) for d in range(nd)] for k in range(nd)]
        self.vol = put(each(det / math.factorial(nd)))

    # -- pointwise physics: q a list of components --------------------------
    def flux(self, q):
        """[d][c]: the flux along each axis."""
        kind, prm = self.p["case"]["problem"], self.p["prm"]
        if kind == "advection":
            return [[v * q[0]] for v in prm["v"]]
        if kind == "cavity":
            z, c2 = torch.zeros_like(q[0]), prm["c"] ** 2
            Ex, Ey, Ez, Bx, By, Bz = q
            return [[z, c2 * Bz, -c2 * By, z, -Ez, Ey], [-c2 * Bz, z, c2 * Bx, Ez, z, -Ex]]
        if kind == "dam_break":
            h = q[0].clamp(min=1e-6)
            u, v, pr = q[1] / h, q[2] / h, 0.5 * prm["g"] * h * h
            return [[q[1], q[1] * u + pr, q[1] * v], [q[2], q[2] * u, q[2] * v + pr]]
        if kind == "alfven":
            r, u, v, p, Bx, By, BB = self._mhd(q)
            E, psi, ps, uB = q[5], q[6], p + 0.5 * BB, u * Bx + v * By
            ch2 = prm["ch"] ** 2
            return [[q[1], q[1] * u + ps - Bx * Bx, q[1] * v - Bx * By, psi, u * By - v * Bx, (E + ps) * u - Bx * uB, ch2 * Bx],
                    [q[2], q[2] * u - By * Bx, q[2] * v + ps - By * By, v * Bx - u * By, psi, (E + ps) * v - By * uB, ch2 * By]]
        r, u, p = self._euler(q)
        out = []
        for d in range(self.nd):
            m = q[1 + d]
            f = [m] + [m * u[k] + (p if k == d else 0) for k in range(3)] + [u[d] * (q[4] + p)]
            out.append(f)
        return out

    def _euler(self, q):
        r = q[0].clamp(min=1e-6)
        u = [m / r for m in q[1:4]]
        p = ((self.p["prm"]["gamma"] - 1) * (q[4] - 0.5 * (q[1] ** 2 + q[2] ** 2 + q[3] ** 2) / r)).clamp(min=1e-6)
        return r, u, p

    def _mhd(self, q):
        r = q[0].clamp(min=1e-6)
        Bx, By = q[3], q[4]
        BB = Bx * Bx + By * By
        p = ((self.p["prm"]["gamma"] - 1) * (q[5] - 0.5 * (q[1] ** 2 + q[2] ** 2) / r - 0.5 * BB)).clamp(min=1e-6)
        return r, q[1] / r, q[2] / r, p, Bx, By, BB

    def _along(self, q):
        F = self.flux(q)
        return [sum(F[d][c] * self.normal[d] for d in range(self.nd)) for c in range(self.NC)]

    def between(self, a, b):
        """The numerical flux from state a to b along the outward normals."""
        kind, prm = self.p["case"]["problem"], self.p["prm"]
        fa, fb, n = self._along(a), self._along(b), self.normal
        if kind == "advection":
            s = abs(sum(v * x for v, x in zip(prm["v"], n)))
        elif kind == "cavity":
            s = prm["c"]
        elif kind == "alfven":
            s = None
            for q in (a, b):
                r, u, v, p, Bx, By, BB = self._mhd(q)
                cs, both = prm["gamma"] * p / r, prm["gamma"] * p / r + BB / r
                fast = torch.sqrt(0.5 * (both + torch.sqrt((both * both - 4 * cs * Bx * Bx / r).clamp(min=0))))
                one = (torch.sqrt(u * u + v * v) + fast).clamp(min=prm["ch"])
                s = one if s is None else torch.maximum(s, one)
        elif kind == "dam_break":
            ha, hb = a[0].clamp(min=1e-6), b[0].clamp(min=1e-6)
            ua, ub = ((q[1] * n[0] + q[2] * n[1]) / h for q, h in ((a, ha), (b, hb)))
            ca, cb = torch.sqrt(prm["g"] * ha), torch.sqrt(prm["g"] * hb)
            return self._hll(a, b, fa, fb, torch.minimum(ua - ca, ub - cb), torch.maximum(ua + ca, ub + cb))
        else:
            return self._euler_between(a, b, fa, fb)
        return [0.5 * (x + y) - 0.5 * s * (v - u) for x, y, u, v in zip(fa, fb, a, b)]

    @staticmethod
    def _hll(a, b, fa, fb, lo, hi):
        lo, hi = lo.clamp(max=0), hi.clamp(min=0)
        return [(hi * x - lo * y + lo * hi * (v - u)) / (hi - lo) for x, y, u, v in zip(fa, fb, a, b)]

    def _euler_between(self, a, b, fa, fb):
        g, n = self.p["prm"]["gamma"], self.normal + [0.0] * (3 - self.nd)
        sides = []
        for q in (a, b):
            r, u, p = self._euler(q)
            sides.append((r, u, p, sum(x * y for x, y in zip(u, n)), torch.sqrt(g * p / r)))
        (ra, ua, pa, na, ca), (rb, ub, pb, nb, cb) = sides
        if self.p["prm"]["flux"] == "rusanov":
            s = torch.maximum(na.abs() + ca, nb.abs() + cb)
            return [0.5 * (x + y) - 0.5 * s * (v - u) for x, y, u, v in zip(fa, fb, a, b)]
        wa, wb = torch.sqrt(ra), torch.sqrt(rb)
        mean = [(wa * x + wb * y) / (wa + wb) for x, y in zip(ua, ub)]
        H = (wa * (a[4] + pa) / ra + wb * (b[4] + pb) / rb) / (wa + wb)
        c = torch.sqrt(((g - 1) * (H - 0.5 * sum(x * x for x in mean))).clamp(min=0))
        m = sum(x * y for x, y in zip(mean, n))
        lo, hi = torch.minimum(na - ca, m - c), torch.maximum(nb + cb, m + c)
        if self.p["prm"]["flux"] == "hlle":
            return self._hll(a, b, fa, fb, lo, hi)
        A, B = ra * (lo - na), rb * (hi - nb)
        mid = (pb - pa + A * na - B * nb) / (A - B)
        left = mid >= 0
        pick = lambda x, y: torch.where(left, x, y)  # noqa: E731
        r, p, un, s, R = pick(ra, rb), pick(pa, pb), pick(na, nb), pick(lo, hi), pick(A, B)
        q, f, u = [pick(x, y) for x, y in zip(a, b)], [pick(x, y) for x, y in zip(fa, fb)], [pick(x, y) for x, y in zip(ua, ub)]
        k = R / (s - mid)
        star = [k] + [k * (u[d] + (mid - un) * n[d]) for d in range(3)] + [k * (q[4] / r + (mid - un) * (mid + p / R))]
        s = pick(s.clamp(max=0), s.clamp(min=0))
        return [x + s * (y - z) for x, y, z in zip(f, star, q)]

    def ghost(self, q):
        """The state behind a boundary: slip or conducting walls, outflow."""
        kind, n = self.p["case"]["problem"], self.normal
        if kind == "advection":
            return [torch.zeros_like(q[0])]
        wall = list(q)
        if kind == "cavity":
            En, Bn = q[0] * n[0] + q[1] * n[1], q[3] * n[0] + q[4] * n[1]
            wall = [2 * En * n[0] - q[0], 2 * En * n[1] - q[1], -q[2], q[3] - 2 * Bn * n[0], q[4] - 2 * Bn * n[1], q[5]]
        else:
            mn = sum(q[1 + d] * n[d] for d in range(self.nd))
            for d in range(self.nd):
                wall[1 + d] = q[1 + d] - 2 * mn * n[d]
        return [torch.where(self.bc_nodes == 1, x, y) for x, y in zip(wall, q)]

    # -- the method ------------------------------------------------------------
    def rate(self, q):
        here = q[self.own]
        there = q.permute(0, 2, 1)[self.nb_n, self.nb_e_nodes]        # [F*NFP, K, NC]
        a, b = [here[:, c] for c in range(self.NC)], [there[..., c] for c in range(self.NC)]
        if self.bcs:
            b = [torch.where(self.bc_nodes > 0, x, y) for x, y in zip(self.ghost(a), b)]
        s = torch.stack([f * self.scale for f in self.between(a, b)], dim=1)
        F = self.flux([q[:, c] for c in range(self.NC)])
        G = torch.cat([torch.stack([sum(self.inv[k][d] * F[d][c] for d in range(self.nd)) for c in range(self.NC)], 1)
                       for k in range(self.nd)], 0)
        flat = lambda x: x.reshape(x.shape[0], -1)  # noqa: E731
        return (self.D @ flat(G) - self.lift @ flat(s)).reshape(q.shape)

    def positive(self, q):
        """The density and pressure floors of the trait Euler equations."""
        g1 = self.p["prm"]["gamma"] - 1
        m2 = (q[:, 1:4] ** 2).sum(1)
        low = ~(q[:, 0] > 1e-6)
        p = g1 * (q[:, 4] - 0.5 * m2 / q[:, 0])
        E = torch.where(p > 1e-6, q[:, 4], 0.5 * m2 / q[:, 0] + 1e-6 / g1)
        q = torch.cat([q[:, :4], E[:, None]], 1)
        rest = torch.zeros_like(q)
        rest[:, 0], rest[:, 4] = 1e-6, 1e-6 / g1
        return torch.where(low[:, None], rest, q)

    def limited(self, q, eps2=0.01):
        """Barth-Jespersen with Venkatakrishnan's function on component 0."""
        mean = torch.tensordot(self.w, q, dims=1)                     # [NC, K]
        m0 = mean[0]
        near = torch.where(self.bc > 0, m0, m0[self.nb_e])
        up = torch.maximum(near.amax(0), m0) - m0
        down = m0 - torch.minimum(near.amin(0), m0)
        d = q[:, 0] - m0
        B, x = torch.where(d > 0, up, down), d.abs()
        g = (B * B + 2 * B * x + eps2) / (B * B + 2 * x * x + B * x + eps2)
        theta = torch.where(x > 1e-30, g, torch.ones_like(g)).amin(0).clamp(max=1)
        return mean + theta * (q - mean)

    def step(self, q, dt):
        kind = self.p["case"]["problem"]
        u = q
        for a, b in ((0.0, 1.0), (0.75, 0.25), (1 / 3, 2 / 3)):
            u = (a * q if a else 0) + b * (u + dt * self.rate(u))
            if kind in ("vortex", "tgv", "sod"):
                u = self.positive(u)
            if kind == "alfven" and a == 1 / 3:
                u[:, 6] *= math.exp(-self.p["prm"]["alpha"] * dt)
            if kind in LIMITED:
                u = self.limited(u)
        return u

    def load(self, q0):
        return torch.as_tensor(q0, device=self.dev).permute(1, 2, 0).contiguous()

    def store(self, q):
        return q.permute(2, 0, 1).contiguous().cpu().numpy()

    def integrals(self, q):
        wv = self.w[:, None] * self.vol
        return dict(integral=(wv[:, None] * q).sum((0, 2)).cpu().numpy(),
                    squared=(wv[:, None] * q * q).sum((0, 2)).cpu().numpy(),
                    maxabs=q.abs().amax((0, 2)).cpu().numpy())

    def energies(self, q):
        """Kinetic energy and enstrophy of an Euler state in three dimensions."""
        wv, r = self.w[:, None] * self.vol, q[:, 0]
        u = [q[:, 1 + d] / r for d in range(3)]
        ref = [[self.nodal[k] @ u[c] for k in range(3)] for c in range(3)]
        grad = [[sum(self.inv[k][d] * ref[c][k] for k in range(3)) for d in range(3)] for c in range(3)]
        curl = [grad[2][1] - grad[1][2], grad[0][2] - grad[2][0], grad[1][0] - grad[0][1]]
        return [float((wv * 0.5 * r * sum(x * x for x in v)).sum()) for v in (u, curl)]


def _seconds(case):
    """About what the reference method takes on the GPU."""
    points = elements(case) * (nodes(dims(case), case["P"]) + (dims(case) + 1) * nodes(2, case["P"]) * (1 if dims(case) == 3 else 0)
                               + 3 * (case["P"] + 1))
    return 3 * case["steps"] * (1.5e-3 + 8e-10 * points)


def exact(case, seed):
    if case["kind"] == "ensemble":
        # the first members stand for all: each is a problem of its own
        members, out = _ensemble(case, seed), []
        for i, p in enumerate(members):
            if i >= 4:
                out.append(None)
                continue
            f = _Field(p)
            q = f.load(p["q0"])
            for _ in range(case["steps"]):
                q = f.step(q, p["dt"])
            out.append(f.store(q))
        return out
    if _seconds(case) > 20:
        return None
    p = _problem(case, seed)
    f = _Field(p)
    q, dt, rows, times = f.load(p["q0"]), p["dt"], [], []
    if case["kind"] == "loop":
        end, t, k = (case["steps"] - 0.5) * dt, 0.0, 1
        frame = end / 4
        while t < end:
            step = min(dt, k * frame - t if k * frame - t > 0 else dt, end - t)
            q = f.step(q, step)
            t += step
            if t >= k * frame - 1e-12 and k <= 4:
                rows.append(f.integrals(q))
                k += 1
        return dict(rows=rows, q=f.store(q))
    for _ in range(case["steps"]):
        if case["kind"] == "adaptive":
            r, u, pr = f._euler([q[:, c] for c in range(5)])
            speed = float((torch.sqrt(sum(x * x for x in u)) + torch.sqrt(GAMMA * pr / r)).max())
            dt = 0.15 * p["h"] / (speed * (2 * case["P"] + 1))
            times.append(dt)
        q = f.step(q, dt)
    if case["kind"] == "adaptive":
        return dict(dt=np.array(times), q=f.store(q))
    if case["problem"] == "tgv":
        return dict(energies=np.array(f.energies(q)), q=f.store(q))
    return f.store(q)
