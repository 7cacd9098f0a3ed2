"""The workloads this framework is timed on: its public entry points at the sizes a user of the
relaxation solver, of the reference's own C functions, of the Einstein Toolkit consumer path and
of the learned initial guess runs them with.

`listed()` names them, `draw(rng)` gives another one of the same ranges, `prepare(case, seed)`
makes what a program holds before the call, `run(state)` is one pass, `work(case)` what a pass
cannot do without, `exact(case, seed)` the pass in plain 64-bit torch, without this package.

Kinds of case:
  operators  rhs_eval, then apply_bcs_outerradiation_and_inner: one substep of a caller who keeps
             their own time integrator (the reference's RHS string)
  loop       the reference driver's main loop on the reference's functions: zero guess, then per
             step residual_all_points, L2_norm_of_gf, MoL_step_forward_in_time
  relax      a resident solver's solve from the zero guess, to a residual target or a step cap
  batch      BatchSolver over configurations on grids of several sizes
  admbase    the solved u to the 17 ADMBase fields at an evolution grid's Cartesian points
  train      a training run of the initial-guess network from given weights
  seed       the network's guess written into a problem's state
"""
from __future__ import annotations

import ctypes as C
import math
from fractions import Fraction
from types import SimpleNamespace

import numpy as np
import torch

from nrpyelliptic_amd import config, mlp, runtime

NG = 5
AMAX, SINHWAA = 1.0e6, 0.07
RADIUS = 100.0                 # integration radius of the residual's L2 norm
SOMMERFELD_SPEED = 4.4793122676309114e+06
TRAIN_SEED, TRAIN_LR = 11, 2.0e-3
WEIGHTS = "nrpyelliptic_amd/data/mlp_initial_guess.npz"
HIDDEN, WIDTH, K0 = 5, 256, 64


def listed():
    return [
        # the smallest call there is: the grid of the smoke test, every call is launch and latency
        dict(name="operators_16x16x6", kind="operators", Nxx="16x16x6", binary="boosted"),
        # the same functions on a grid no tile width divides
        dict(name="operators_200x130x16", kind="operators", Nxx="200x130x16", binary="unequal"),
        # the reference's main.c relinked against this library, at the production size
        dict(name="loop_128x128x16", kind="loop", Nxx="128x128x16", binary="boosted", steps=10),
        # the small axisymmetric spinning case, solved to the end
        dict(name="relax_64x64x4", kind="relax", Nxx="64x64x4", binary="axisymmetric", precision=64,
             outer_bc="radiation", cfl=0.7, target=-10.0, steps=2407, cap=20000),
        # the production solve: 128x128x16 in FP64 from the zero guess to log10 L2 <= -10
        dict(name="relax_128x128x16", kind="relax", Nxx="128x128x16", binary="boosted", precision=64,
             outer_bc="radiation", cfl=0.7, target=-10.0, steps=3144, cap=20000),
        # FP32 bulk, FP64 finish: unequal masses with spins
        dict(name="mixed_128x128x16", kind="relax", Nxx="128x128x16", binary="q4", precision=32,
             outer_bc="radiation", cfl=0.7, target=-10.0, steps=4241, cap=20000),
        # the Einstein Toolkit thorn's outer boundary condition on its default grid
        dict(name="sommerfeld_128x128x16", kind="relax", Nxx="128x128x16", binary="boosted", precision=64,
             outer_bc="sommerfeld6", cfl=0.7, target=-10.0, steps=400, cap=400),
        # a large single grid (the first part of its relaxation)
        dict(name="relax_256x256x32", kind="relax", Nxx="256x256x32", binary="boosted", precision=64,
             outer_bc="radiation", cfl=0.7, target=-10.0, steps=200, cap=200),
        # a slice of the 64-configuration batch: mixed grids, relaxed together
        dict(name="batch_16", kind="batch", cfl=0.5, steps=200, grids=" ".join(
            ["96x96x8", "128x128x16", "160x128x16", "96x128x8", "128x96x16", "160x96x8", "96x96x16", "128x128x8"] * 2)),
        # ADMBase fields on a 128^3 evolution grid, the thorn's default interpolation order
        dict(name="admbase_128x128x128", kind="admbase", Nxx="128x128x16", binary="boosted", points="128x128x128",
             order=4, plane=0, lapse=0),
        # the initial-guess network's training loop at its production minibatch
        dict(name="train_8192", kind="train", rows=65536, batch=8192, steps=100),
        # its use: features, inference and smoothing on the production grid
        dict(name="seed_128x128x16", kind="seed", Nxx="128x128x16", binary="boosted", smooth=2),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["operators", "loop", "relax", "relax", "batch", "admbase", "train", "seed"])

    def grid(points, n2s=(2, 4, 6, 8, 10, 12, 16, 24, 32)):
        while True:
            n = (_log_int(rng, 12, 320), 2 * _log_int(rng, 6, 140), rng.choice(n2s))  # Nxx1, Nxx2 are even on this grid
            if n[0] * n[1] * n[2] <= points:
                return "%dx%dx%d" % n

    binary = rng.choice(["boosted", "unequal"])
    if kind == "operators":
        return dict(kind=kind, Nxx=grid(2 << 20), binary=binary)
    if kind == "loop":
        return dict(kind=kind, Nxx=grid(2 << 20), binary=binary, steps=rng.randint(2, 12))
    if kind == "relax":
        steps = 50 * rng.randint(1, 4)
        return dict(kind=kind, Nxx=grid(2 << 20), binary=binary, precision=rng.choice([64, 64, 32]),
                    outer_bc=rng.choice(["radiation", "radiation", "sommerfeld6"]), cfl=0.5, target=-10.0,
                    steps=steps, cap=steps)
    if kind == "batch":
        return dict(kind=kind, cfl=0.5, steps=50 * rng.randint(1, 4),
                    grids=" ".join(grid(400000, (4, 6, 8, 12, 16)) for _ in range(rng.randint(2, 12))))
    if kind == "admbase":
        return dict(kind=kind, Nxx=grid(1 << 20, (8, 12, 16)), binary=binary, order=rng.randint(1, 6),
                    points="%dx%dx%d" % tuple(_log_int(rng, 8, 128) for _ in range(3)), plane=rng.randint(0, 1),
                    lapse=rng.randint(0, 1))
    if kind == "train":
        return dict(kind=kind, rows=rng.randint(5000, 70000), batch=64 * _log_int(rng, 4, 128),
                    steps=rng.randint(10, 100))
    return dict(kind=kind, Nxx=grid(1 << 20, (6, 8, 12, 16)), binary=binary, smooth=rng.randint(0, 3))


# --- inputs, made from the seed alone -----------------------------------------------------------

def _dims(text):
    return tuple(int(n) for n in text.split("x"))


def _binary(kind, rng):
    """Puncture parameters around the package's own configurations."""
    base = dict(bare_mass=(0.5, 0.5), pos0=(0.0, 0.0, 5.0), pos1=(0.0, 0.0, -5.0), P0=(0.0,) * 3, P1=(0.0,) * 3,
                S0=(0.0,) * 3, S1=(0.0,) * 3, bScale=5.0, eta=20.0, AMAX=AMAX, SINHWAA=SINHWAA)
    if kind == "axisymmetric":
        return dict(base, S0=(0.0, 0.0, 0.2 * rng.uniform(0.9, 1.1)), S1=(0.0, 0.0, 0.2 * rng.uniform(0.9, 1.1)))
    if kind == "boosted":
        P = 0.0953 * rng.uniform(0.97, 1.03)
        return dict(base, P0=(0.0, P, 0.0), P1=(0.0, -P, 0.0))
    q, D = (4.0, 10.0) if kind == "q4" else (rng.uniform(1.2, 5.0), rng.uniform(8.0, 12.0))
    m0, m1 = q / (1.0 + q), 1.0 / (1.0 + q)
    P = m0 * m1 / math.sqrt(D)
    S = []
    for m in (m0, m1):
        v = rng.normal(size=3)
        S.append(tuple(float(x) for x in v / np.linalg.norm(v) * rng.uniform(0.0, 0.6) * m * m))
    return dict(base, bare_mass=(m0, m1), pos0=(0.0, 0.0, D / 2), pos1=(0.0, 0.0, -D / 2), P0=(0.0, P, 0.0),
                P1=(0.0, -P, 0.0), S0=S[0], S1=S[1], bScale=D / 2)


def _configs(case, seed):
    rng = np.random.default_rng(seed)
    grids = case["grids"].split() if case["kind"] == "batch" else [case["Nxx"]]
    return [SimpleNamespace(Nxx=_dims(g), CFL=case.get("cfl", 0.7), **_binary(case.get("binary", "unequal"), rng))
            for g in grids]


def _state_input(grid, seed):
    """A state as a caller's integrator holds it mid-relaxation: u about the size and falloff of a
    solution, v near eta u, rough at the level of a part in a thousand, ghosts at their images."""
    rng = np.random.default_rng(seed + 7919)
    shape = (grid.N[2], grid.N[1], grid.N[0] + NG)
    rough = 1.0 + 1e-3 * torch.from_numpy(rng.uniform(-1.0, 1.0, (2,) + shape)).to(grid.dev)
    r = grid.radius()[:, NG:].expand(shape)
    u = 0.05 / (1.0 + r / 5.0) * rough[0]
    return torch.stack([grid.pad(u), grid.pad(20.0 * u * rough[1])])


def _points(case, seed):
    rng = np.random.default_rng(seed + 31)
    c = rng.uniform(-0.5, 0.5, 3)
    ax = [np.linspace(-20.0, 20.0, n) + o for n, o in zip(_dims(case["points"]), c)]
    z, y, x = np.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    return x.ravel(), y.ravel(), z.ravel()


def _dataset(case, seed):
    """Feature rows in the ranges the features have (23 used, zero-padded to 64, BF16) and smooth
    targets of them; He-initialised weights."""
    rng = np.random.default_rng(seed)
    X = np.zeros((case["rows"], K0), np.float32)
    X[:, :23] = rng.uniform(-1.0, 1.0, (case["rows"], 23))
    X = torch.from_numpy(X).bfloat16().float().numpy()
    t = (np.sin(2.0 * X[:, 0] + X[:, 3]) + 0.5 * X[:, 1] * X[:, 2] - 0.3 * X[:, 7]).astype(np.float32)
    p = []
    for l in range(1, HIDDEN + 2):
        fan, n = (23 if l == 1 else WIDTH), (1 if l > HIDDEN else WIDTH)
        a = math.sqrt(6.0 / fan) * (0.1 if l > HIDDEN else 1.0)
        p += [rng.uniform(-a, a, n * (K0 if l == 1 else WIDTH)), np.zeros(n)]
    return X, t, np.concatenate(p).astype(np.float32)


# --- the pass -----------------------------------------------------------------------------------

class _Held:
    """What a state has on the device. Every view of it holds it too, so that an output outlives
    the state it came from."""

    def __init__(self):
        self.close_me, self.arrays = [], []

    def __del__(self):
        for o in self.close_me:
            o.close()


class _View:
    """Device memory of the library as torch sees it."""

    def __init__(self, held, ptr, n):
        self.held = held
        self.__cuda_array_interface__ = dict(shape=(n,), typestr="<f8", data=(C.cast(ptr, C.c_void_p).value, False),
                                             version=2, strides=None)


def _view(held, ptr, n):
    t = torch.as_tensor(_View(held, ptr, n), device="cuda")
    t.held = held
    return t


def prepare(case, seed):
    s, held = SimpleNamespace(case=case), _Held()
    s.held = held
    kind = case["kind"]

    def array(n, dtype=np.float64):
        held.arrays.append(runtime.DeviceArray(n, dtype))
        return held.arrays[-1]

    if kind == "train":
        X, t, s.p0 = _dataset(case, seed)
        s.X = array(X.size, np.uint16).upload(mlp.bf16_bits(X).ravel())
        s.t = array(t.size, np.float32).upload(t)
        return s
    s.probs = [runtime.Problem(config.PunctureConfig(**vars(c))) for c in _configs(case, seed)]
    held.close_me = list(s.probs)
    P = s.probs[0]
    s.y = [_view(held, Q.gd.gridfuncs.y_n_gfs, 2 * Q.ntot) for Q in s.probs]
    if kind == "relax":
        s.solver = P.solver(precision=case["precision"], outer_bc=case["outer_bc"], log10_target=case["target"],
                            max_steps=case["cap"])
        held.close_me.insert(0, s.solver)
    elif kind == "batch":
        s.solver = runtime.BatchSolver(s.probs, max_steps=case["steps"])
        held.close_me.insert(0, s.solver)
    elif kind == "operators":
        s.y[0].copy_(_state_input(_Grid(_configs(case, seed)[0]), seed).reshape(-1))
        s.dev = array(2 * P.ntot).upload(np.zeros(2 * P.ntot))
        s.rhs = _view(held, s.dev.ptr, 2 * P.ntot)
        p = P.gd.params
        s.speed = (C.c_double * 2)(p.uu_wavespeed_at_OB, p.vv_wavespeed_at_OB)
        s.finf = (C.c_double * 2)(0.0, 0.0)
    elif kind == "admbase":
        s.y[0].copy_(_state_input(_Grid(_configs(case, seed)[0]), seed).reshape(-1))
        pts = _points(case, seed)
        n = pts[0].size
        s.xyz = [array(n).upload(a) for a in pts]
        s.outs = [array(n) for _ in runtime.ADMBASE_NAMES]
        s.fields = [_view(held, d.ptr, n) for d in s.outs]
        s.lsh = (C.c_int * 3)(*_dims(case["points"]))
        o = s.opt = runtime.admbase_options()
        o.orbital_plane, o.initial_lapse, o.lapse_exponent_n = case["plane"], case["lapse"], -2.0
        o.NRPy_epsilon, o.interpolation_order = 1e-8, case["order"]
    elif kind == "seed":
        s.net = mlp.InitialGuessMLP()
        s.net.load(WEIGHTS)
        held.close_me.append(s.net)
    torch.cuda.synchronize()
    return s


def run(s):
    case, kind, L = s.case, s.case["kind"], runtime.lib()
    if kind == "train":
        net = mlp.InitialGuessMLP()
        net.set_params(s.p0)
        losses = net.train(s.X, s.t, case["rows"], case["batch"], case["steps"], TRAIN_LR, seed=TRAIN_SEED)
        p = net.get_params()
        net.close()
        return {"params": p, "losses": losses}
    P = s.probs[0]
    gd, p = P.gd, C.byref(P.gd.params)
    gf = gd.gridfuncs
    if kind == "operators":
        out = s.dev.as_real_p()
        L.rhs_eval(p, C.byref(gd.rfmstruct), gf.auxevol_gfs, gf.y_n_gfs, out)
        L.apply_bcs_outerradiation_and_inner(p, C.byref(gd.bcstruct), gd.xx, C.byref(s.speed), C.byref(s.finf),
                                             gf.y_n_gfs, out)
        return {"rhs": s.rhs}
    if kind == "loop":
        P.zero_guess()
        l2 = []
        for _ in range(case["steps"]):
            l2.append(P.log10_residual())
            P.mol_step()
        return {"y": s.y[0], "log10_l2": np.array(l2)}
    if kind == "relax":
        P.zero_guess()
        r = s.solver.solve()
        return {"y": s.y[0], "log10_l2": r.log10_l2, "steps": r.steps}
    if kind == "batch":
        for Q in s.probs:
            Q.zero_guess()
        res, _ = s.solver.solve()
        return {"y": list(s.y), "log10_l2": np.array([r.log10_l2 for r in res]), "steps": [r.steps for r in res]}
    if kind == "admbase":
        runtime.check(L.nrpyell_Initialize_ADMBase(C.byref(gd), C.byref(s.opt), s.lsh, *[d.as_real_p() for d in s.xyz],
                                                   *[d.as_real_p() for d in s.outs]), "Initialize_ADMBase")
        return {"fields": list(s.fields)}
    s.net.seed(P, case["smooth"])
    return {"y": s.y[0]}


# --- what a pass cannot do without --------------------------------------------------------------

# per interior point: the stencil of u (three second and two first 10th-order differences), the
# source term and their sum; an RK4 stage update of u and v
RHS_FLOPS, STAGE_FLOPS = 95.0, 8.0


def work(case):
    kind = case["kind"]
    if kind == "train":
        flops = 6.0 * case["batch"] * (K0 * WIDTH + (HIDDEN - 1) * WIDTH * WIDTH + WIDTH)
        n = (K0 + 1) * WIDTH + (HIDDEN - 1) * (WIDTH + 1) * WIDTH + WIDTH + 1
        # per step: the minibatch's rows; weights and two Adam moments read and written
        return {"bytes": case["steps"] * (case["batch"] * (2.0 * K0 + 4.0) + 24.0 * n), "flops": case["steps"] * flops}
    n = [math.prod(_dims(g)) for g in (case["grids"].split() if kind == "batch" else [case["Nxx"]])]
    if kind == "operators":  # u, v, three background fields in, two right-hand sides out
        return {"bytes": 56.0 * n[0], "flops": (RHS_FLOPS + 2.0) * n[0]}
    if kind == "admbase":
        m, k = math.prod(_dims(case["points"])), case["order"] + 1
        # x, y, z in, 17 fields out, u once; the molecule's sums and the closed forms
        return {"bytes": 160.0 * m + 8.0 * n[0], "flops": m * (2.0 * k ** 3 + 400.0)}
    if kind == "seed":
        flops = 2.0 * (K0 * WIDTH + (HIDDEN - 1) * WIDTH * WIDTH + WIDTH) + 100.0
        return {"bytes": 16.0 * n[0], "flops": flops * n[0]}
    # per RK4 step: u, v in and out, psi and AA^2 in; four substeps
    size = 4.0 if case.get("precision") == 32 else 8.0
    return {"bytes": 6.0 * size * case["steps"] * sum(n),
            "flops": 4.0 * (RHS_FLOPS + STAGE_FLOPS) * case["steps"] * sum(n)}


# --- the pass in plain 64-bit torch -------------------------------------------------------------

def _fd_weights(nodes, deriv):
    """Weights of the deriv-th derivative at 0 on integer nodes (exact rational solve)."""
    n = len(nodes)
    A = [[Fraction(x) ** k for x in nodes] + [Fraction(math.factorial(k) if k == deriv else 0)] for k in range(n)]
    for c in range(n):
        p = next(r for r in range(c, n) if A[r][c] != 0)
        A[c], A[p] = A[p], A[c]
        A[c] = [a / A[c][c] for a in A[c]]
        for r in range(n):
            if r != c and A[r][c] != 0:
                A[r] = [a - A[r][c] * b for a, b in zip(A[r], A[c])]
    return [float(A[k][n]) for k in range(n)]


class _Grid:
    """The prolate-spheroidal (SinhSymTP) grid: independent points are i0 = NG .. N0+2NG-1 (five
    outer layers), i1 and i2 interior; fields are [i2, i1, i0]."""

    def __init__(self, cfg):
        self.dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        self.cfg, self.N = cfg, tuple(cfg.Nxx)
        self.dx = (1.0 / self.N[0], math.pi / self.N[1], 2.0 * math.pi / self.N[2])
        self.x = [torch.arange(-NG, n + NG, dtype=torch.float64, device=self.dev).add(0.5).mul(d).add(o)
                  for n, d, o in zip(self.N, self.dx, (0.0, 0.0, -math.pi))]
        w, b = cfg.SINHWAA, cfg.bScale
        A = cfg.AMAX / math.sinh(1.0 / w)
        self.r, self.rp = A * torch.sinh(self.x[0] / w), A / w * torch.cosh(self.x[0] / w)  # f0, f0'
        self.rpp = self.r / w ** 2
        self.sin, self.cos = torch.sin(self.x[1])[:, None], torch.cos(self.x[1])[:, None]
        self.F = self.r ** 2 + (b * self.sin) ** 2
        self.f3sq = self.r ** 2 + b * b

    def radius(self):
        return torch.sqrt(self.r ** 2 + (self.cfg.bScale * self.cos[NG:-NG]) ** 2)

    def pad(self, f):
        """All ghost points from the independent ones: reflections carry a half turn in phi."""
        h = self.N[2] // 2
        f = torch.cat([torch.roll(f[:, :, :NG].flip(2), h, 0), f], 2)
        f = torch.cat([torch.roll(f[:, :NG].flip(1), h, 0), f, torch.roll(f[:, -NG:].flip(1), h, 0)], 1)
        j = torch.arange(-NG, self.N[2] + NG, device=self.dev) % self.N[2]
        return f[j]


class _Relaxation:
    """The relaxation system on a _Grid: du/dt = v - eta u, dv/dt = c^2 (lap u + AA/(8 (psi+u)^7)),
    an outgoing condition on the outer layers, RK4."""

    def __init__(self, cfg, outer_bc="radiation"):
        g = self.g = _Grid(cfg)
        self.outer_bc, self.eta = outer_bc, cfg.eta
        I0, I1 = slice(NG, -NG), slice(NG, -NG)
        b, sin, cos = cfg.bScale, g.sin[I1], g.cos[I1]
        r, rp, rpp, F, f3sq = g.r[I0], g.rp[I0], g.rpp[I0], g.F[I1, I0], g.f3sq[I0]
        self.K = (f3sq / (F * rp ** 2), (1.0 / F), 1.0 / (r * sin) ** 2, cos / sin / F,
                  ((2.0 * r + b * b / r) / rp - f3sq * rpp / rp ** 3) / F)
        ds = torch.stack([g.dx[0] * rp * torch.sqrt(F / f3sq), g.dx[1] * torch.sqrt(F), g.dx[2] * r * sin])
        self.dt = float(ds.min())
        c = cfg.CFL * ds.min(0).values / self.dt
        self.c2, self.c_out = c * c, float(c[0, -1])
        w = r * rp * F * sin / torch.sqrt(f3sq) * math.prod(g.dx)
        self.w = torch.where(torch.sqrt(r ** 2 + (b * cos) ** 2) < RADIUS, w, torch.zeros_like(w))
        self.volume = float(self.w.sum()) * g.N[2]
        self.psi, self.AA = self.background()
        # the last interior column and the outer layers: R, dx0/dR, dx1/dR
        e0 = slice(g.N[0] + NG - 1, g.N[0] + 2 * NG)
        re = g.r[e0]
        self.R = torch.sqrt(re ** 2 + (b * cos) ** 2)
        Fe = g.F[I1, e0]
        self.g0 = re * g.f3sq[e0] / (Fe * g.rp[e0] * self.R)
        self.g1 = -b * b * sin * cos / (Fe * self.R)
        c5 = list(range(-5, 6))
        self.w1, self.w2 = _fd_weights(c5, 1), _fd_weights(c5, 2)
        if outer_bc == "radiation":
            self.edge = [[(k, v) for k, v in zip(nodes, _fd_weights(nodes, 1))]
                         for nodes in (list(range(-5 - max(1, q), 6 - max(1, q))) for q in range(6))]
        else:
            back = [(-k, -v) for k, v in enumerate(_fd_weights(list(range(7)), 1))]
            self.edge = [back] * 6
            self.c_out = SOMMERFELD_SPEED

    def background(self):
        g, cfg = self.g, self.g.cfg
        x0, x1, x2 = g.x[0][NG:-NG], g.x[1][NG:-NG, None], g.x[2][NG:-NG, None, None]
        rho = g.r[NG:-NG] * torch.sin(x1)
        X = [rho * torch.cos(x2), rho * torch.sin(x2), (torch.sqrt(g.f3sq[NG:-NG]) * torch.cos(x1)).expand(rho.shape)]
        h, A = _bowen_york(cfg, [a.expand(g.N[2], *rho.shape) for a in X], range(3))
        return 1.0 + h, sum(A[min(i, j), max(i, j)] ** 2 for i in range(3) for j in range(3))

    def diff(self, p, axis, weights):
        """Sum of weights at offsets -5 .. 5 along an axis of a padded field, at the interior."""
        out = 0.0
        for k, w in zip(range(-5, 6), weights):
            s = [slice(NG, -NG)] * 3
            s[axis] = slice(NG + k, p.shape[axis] - NG + k)
            out = out + w * p[tuple(s)] if w else out
        return out

    def residual(self, p):
        dx = self.g.dx
        u = p[NG:-NG, NG:-NG, NG:-NG]
        return (self.K[0] * self.diff(p, 2, self.w2) / dx[0] ** 2 + self.K[1] * self.diff(p, 1, self.w2) / dx[1] ** 2
                + self.K[2] * self.diff(p, 0, self.w2) / dx[2] ** 2 + self.K[3] * self.diff(p, 1, self.w1) / dx[1]
                + self.K[4] * self.diff(p, 2, self.w1) / dx[0] + self.AA / (8.0 * (self.psi + u) ** 7))

    def log10_l2(self, y):
        return float(torch.log10(1e-16 + torch.sqrt((self.w * self.residual(self.g.pad(y[0])) ** 2).sum() / self.volume)))

    def outgoing(self, f):
        """-c (d_R f + f / R) at the last interior column and the outer layers of a field."""
        g, n0 = self.g, self.g.N[0]
        p = g.pad(f)
        cols = p[NG:-NG, NG:-NG]
        d0 = torch.stack([sum(w * cols[:, :, n0 + NG - 1 + q + k] for k, w in self.edge[q]) for q in range(6)], 2)
        e = p[NG:-NG, :, n0 + NG - 1:]
        n1 = g.N[1]
        if self.outer_bc == "radiation":
            d1 = sum(w * e[:, NG + k:NG + k + n1] for k, w in zip(range(-5, 6), self.w1) if w)
        else:
            d1 = sum(w * e[:, NG + k:NG + k + n1] for k, w in zip(range(-3, 4), _fd_weights(list(range(-3, 4)), 1)) if w)
            d1[:, 0] = sum(w * e[:, NG + k] for k, w in enumerate(_fd_weights(list(range(7)), 1)))
        f = cols[:, :, n0 + NG - 1:]
        return -self.c_out * (self.g0 * d0 / g.dx[0] + self.g1 * d1 / g.dx[1] + f / self.R)

    def rhs(self, y):
        n0 = self.g.N[0]
        k = torch.empty_like(y)
        k[0, :, :, :n0] = y[1, :, :, :n0] - self.eta * y[0, :, :, :n0]
        k[1, :, :, :n0] = self.c2 * self.residual(self.g.pad(y[0]))
        for f in range(2):
            A = self.outgoing(y[f])
            q = (self.R[:, :1] / self.R[:, 1:]) ** 3
            k[f, :, :, n0:] = A[:, :, 1:] + q * (k[f, :, :, n0 - 1:n0] - A[:, :, :1])
        return k

    def step(self, y):
        k1 = self.rhs(y)
        k2 = self.rhs(y + 0.5 * self.dt * k1)
        k3 = self.rhs(y + 0.5 * self.dt * k2)
        k4 = self.rhs(y + self.dt * k3)
        return y + self.dt / 6.0 * (k1 + 2.0 * (k2 + k3) + k4)

    def zero(self):
        g = self.g
        return torch.zeros(2, g.N[2], g.N[1], g.N[0] + NG, dtype=torch.float64, device=g.dev)

    def relax(self, target, cap):
        """Check, stop or step, as the resident solver does; (state, last residual, steps)."""
        y = self.zero()
        for n in range(cap):
            l = self.log10_l2(y)
            if l <= target:
                return y, l, n
            y = self.step(y)
        return y, l, cap

    def full(self, y):
        return torch.stack([self.g.pad(f) for f in y]).reshape(-1)


def _bowen_york(cfg, X, axes):
    """Sum of m/(2 r) and the Bowen-York curvature of both punctures at X; `axes` says which of
    the punctures' own axes the directions of X are."""
    axes = list(axes)
    h, A = 0.0, {}
    for m, pos, P, S in ((cfg.bare_mass[0], cfg.pos0, cfg.P0, cfg.S0), (cfg.bare_mass[1], cfg.pos1, cfg.P1, cfg.S1)):
        pos, P, S = ([v[a] for a in axes] for v in (pos, P, S))
        x = [X[d] - pos[d] for d in range(3)]
        r = (x[0] ** 2 + x[1] ** 2 + x[2] ** 2) ** 0.5
        xP = sum(x[d] * P[d] for d in range(3))
        xS = [x[1] * S[2] - x[2] * S[1], x[2] * S[0] - x[0] * S[2], x[0] * S[1] - x[1] * S[0]]
        h = h + m / (2.0 * r)
        for i in range(3):
            for j in range(i, 3):
                t = 1.5 * (P[i] * x[j] + P[j] * x[i]) / r ** 3 + 1.5 * xP * x[i] * x[j] / r ** 5 \
                    - 3.0 * (xS[i] * x[j] + xS[j] * x[i]) / r ** 5
                if i == j:
                    t = t - 1.5 * xP / r ** 3
                A[i, j] = A[i, j] + t if (i, j) in A else t
    return h, A


def _exact_admbase(case, seed):
    cfg = _configs(case, seed)[0]
    g = _Grid(cfg)
    u = _state_input(g, seed)[0]
    etk = [torch.from_numpy(a).to(g.dev) for a in _points(case, seed)]
    x, y, z = (etk[1], etk[2], etk[0]) if case["plane"] == 0 else etk
    b2 = cfg.bScale ** 2
    R2 = x * x + y * y + z * z
    Q = torch.sqrt(-4.0 * z * z * b2 + b2 * b2 + 2.0 * b2 * R2 + R2 * R2)
    xx = [SINHWAA * torch.asinh(math.sqrt(0.5) * torch.sqrt(-b2 + R2 + Q) * math.sinh(1.0 / SINHWAA) / AMAX),
          torch.acos(0.99999999 * math.sqrt(0.5) * torch.sqrt(R2 / b2 - Q / b2 + 1.0) * torch.sign(z)), torch.atan2(y, x)]
    n = case["order"]
    first, wt = [], []
    for d in range(3):  # centred molecule, moved inward at the array's ends; Lagrange weights
        fp = (xx[d] - g.x[d][0]) / g.dx[d]
        c = torch.floor(fp + (0.5 if n % 2 == 0 else 0.0)) - n // 2
        c = torch.clamp(c, 0, g.x[d].numel() - 1 - n)
        t = fp - c
        wt.append([math.prod([(t - k) / (m - k) for k in range(n + 1) if k != m]) for m in range(n + 1)])
        first.append(c.long())
    flat, G = u.reshape(-1), [a.numel() for a in g.x]
    val = 0.0
    for k in range(n + 1):
        for j in range(n + 1):
            row = first[0] + G[0] * (first[1] + j + G[1] * (first[2] + k))
            val = val + wt[2][k] * wt[1][j] * sum(wt[0][i] * flat[row + i] for i in range(n + 1))
    h, A = _bowen_york(cfg, etk, (2, 0, 1) if case["plane"] == 0 else (0, 1, 2))
    psi = 1.0 + h + val
    lapse = psi ** -2.0 if case["lapse"] == 0 else 0.5 * (1.0 - h) / (1.0 + h) + 0.5
    o = torch.zeros_like(val)
    K = [A[i, j] / psi ** 2 for i in range(3) for j in range(i, 3)]
    return {"fields": [val, lapse, o, o, o, psi ** 4, o, o, psi ** 4, o, psi ** 4] + K}


def _unpack(p):
    out, o = [], 0
    for l in range(1, HIDDEN + 2):
        n, k = (1 if l > HIDDEN else WIDTH), (K0 if l == 1 else WIDTH)
        out.append((p[o:o + n * k].view(n, k), p[o + n * k:o + n * k + n]))
        o += n * k + n
    return out


def _network(p, x):
    for W, b in _unpack(p)[:-1]:
        z = x @ W.T + b
        x = z * torch.sigmoid(z)
    W, b = _unpack(p)[-1]
    return (x @ W.T + b)[:, 0]


def _exact_train(case, seed):
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    X, t, p = (torch.from_numpy(a).to(dev, torch.float64) for a in _dataset(case, seed))
    m, v = torch.zeros_like(p), torch.zeros_like(p)
    mask, losses = (1 << 64) - 1, []
    for k in range(case["steps"]):
        z = np.arange(1, case["batch"] + 1, dtype=np.uint64) * np.uint64(0x9E3779B97F4A7C15)
        z += np.uint64((TRAIN_SEED + 0x632BE59BD9B4E019 * (k + 1)) & mask)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        rows = torch.from_numpy(((z ^ (z >> np.uint64(31))) % np.uint64(case["rows"])).astype(np.int64)).to(dev)
        q = p.clone().requires_grad_(True)
        loss = ((_network(q, X[rows]) - t[rows]) ** 2).mean()
        g, = torch.autograd.grad(loss, q)
        losses.append(float(loss.detach()))
        frac = k / (case["steps"] - 1) if case["steps"] > 1 else 0.0
        lr = TRAIN_LR * (0.01 + 0.99 * 0.5 * (1.0 + math.cos(math.pi * frac)))
        m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
        p = p - lr * (m / (1.0 - 0.9 ** (k + 1))) / (torch.sqrt(v / (1.0 - 0.999 ** (k + 1))) + 1e-8)
    return {"params": p, "losses": np.array(losses)}


def _exact_seed(case, seed):
    cfg = _configs(case, seed)[0]
    g = _Grid(cfg)
    shape = (g.N[2], g.N[1], g.N[0] + NG)
    r, x1, x2 = g.r[NG:], g.x[1][NG:-NG, None], g.x[2][NG:-NG, None, None]
    X = [(r * torch.sin(x1) * torch.cos(x2)).expand(shape), (r * torch.sin(x1) * torch.sin(x2)).expand(shape),
         (torch.sqrt(g.f3sq[NG:]) * torch.cos(x1)).expand(shape)]
    b = cfg.bScale
    R = torch.sqrt(X[0] ** 2 + X[1] ** 2 + X[2] ** 2)
    rn = [torch.sqrt(sum((X[d] - q[d]) ** 2 for d in range(3))) for q in (cfg.pos0, cfg.pos1)]
    f = [a / (R + b) for a in X] + [R / (R + b), torch.log1p(R / b) / 10.0, b / (rn[0] + b), b / (rn[1] + b)]
    f += [*cfg.bare_mass, math.dist(cfg.pos0, cfg.pos1) / 20.0]
    f += [10.0 * a for a in (*cfg.P0, *cfg.P1)]
    f += [a / m ** 2 for m, S in zip(cfg.bare_mass, (cfg.S0, cfg.S1)) for a in S] + [b / 10.0]
    f = torch.stack([a if torch.is_tensor(a) else torch.full(shape, a, dtype=torch.float64, device=g.dev) for a in f], 3)
    with np.load(WEIGHTS, allow_pickle=False) as d:
        p = torch.from_numpy(d["params"]).to(g.dev, torch.float64)
    f = torch.nn.functional.pad(f.reshape(-1, f.shape[3]), (0, K0 - f.shape[3]))
    t = torch.cat([_network(p, c) for c in f.split(1 << 16)]).reshape(shape)
    u = torch.exp(t) / (50.0 * (R + b))
    for _ in range(case["smooth"]):  # binomial smoothing of the interior along i0, i1, i2
        for axis in (2, 1, 0):
            q = g.pad(u)
            s = [slice(NG, -NG)] * 3
            lo, hi = list(s), list(s)
            lo[axis], hi[axis] = slice(NG - 1, -NG - 1), slice(NG + 1, q.shape[axis] - NG + 1)
            u = u.clone()
            u[:, :, :g.N[0]] = 0.25 * (q[tuple(lo)] + q[tuple(hi)]) + 0.5 * q[tuple(s)]
    return {"y": torch.stack([g.pad(u), g.pad(cfg.eta * u)]).reshape(-1)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "admbase":
        return _exact_admbase(case, seed)
    if kind == "train":
        return _exact_train(case, seed)
    if kind == "seed":
        return _exact_seed(case, seed)
    cfgs = _configs(case, seed)
    if kind == "operators":
        R = _Relaxation(cfgs[0])
        y = _state_input(R.g, seed)[:, NG:-NG, NG:-NG, NG:]
        return {"rhs": R.full(R.rhs(y))}
    if kind == "loop":
        R = _Relaxation(cfgs[0])
        y, l2 = R.zero(), []
        for _ in range(case["steps"]):
            l2.append(R.log10_l2(y))
            y = R.step(y)
        return {"y": R.full(y), "log10_l2": np.array(l2)}
    if kind == "batch":
        out = []
        for c in cfgs:
            R = _Relaxation(c)
            y, l, _ = R.relax(-10.0, case["steps"])
            out.append((R.full(y), l))
        return {"y": [o[0] for o in out], "log10_l2": np.array([o[1] for o in out]), "steps": None}
    R = _Relaxation(cfgs[0], case["outer_bc"])
    if case["precision"] == 32 and case["steps"] < case["cap"]:
        # where a mixed solve stops depends on its FP32 phase: the state has no 64-bit value
        return None
    y, l, _ = R.relax(case["target"], case["cap"])
    return {"y": R.full(y), "log10_l2": l, "steps": None}
