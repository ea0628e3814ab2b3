"""Timed workloads of the UGKS time step, through the package's public entry points.

A case is a dict of plain values.  Its geometry, velocity set, scheme and boundary conditions come from
``pyugks_amd.cases`` (the workloads of bench.py and the tests, with odd sizes beside them); the initial flow is a
smooth field of random Fourier modes drawn from the seed.  A pass loads that initial state into the simulation's
device buffers and advances it by ``steps`` time steps, which is what a parameter study or an ensemble of runs does
over and over; it keeps every pass at the same point of the flow (the reference's WENO5 scheme ends in NaN on the
cavities after a hundred steps or so, whatever the precision).

``entry`` names the way a program steps a case:

* ``plan``     StepPlan.run, eager launches
* ``graph``    StepPlan(graph=True).run, replays of the captured step
* ``noalloc``  ugks_step_run_noalloc, the step without device allocations (C entry point)
* ``one_step`` UGKSim.one_step, the per-kernel drop-in path with its host readbacks (FP64)

``exact`` restates the step in torch in 64 bits on the undivided domain, without the package's code.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from pyugks_amd import bc as bcd
from pyugks_amd import cases as wl
from pyugks_amd import lib as L
from pyugks_amd.fused import StepPlan, plan_inputs
from pyugks_amd.sim import UGKSim

METHODS = ("vanLeer", "WENO5", "minmod")
BATCH_SIDES = (32, 64, 96, 128, 192, 256)      # the 64-case batch's sizes and velocity grids
BATCH_GRIDS = (16, 24, 32, 40)
MAX_UPDATES = 6.3e8                            # cell-velocity updates per step of the largest listed case


# ------------------------------------------------------------------ cases --
def _cavity(name, ni, nj, vel, nv, method, Kn, precision, entry, steps, nbi=1, nbj=1, bend=0.0, CFL=0.8):
    c = dict(kind="cavity", ni=ni, nj=nj, nbi=nbi, nbj=nbj, vel=vel, nv=nv, method=method, Kn=Kn, CFL=CFL, bend=bend,
             precision=precision, entry=entry, steps=steps)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smoke test's cavity, two joined blocks: a program that steps tiny cases waits for launches, not for data
        _cavity("tiny_cavity_plan_fp64", 12, 10, "NC", 12, "WENO5", 0.075, "fp64", "plan", 4, nbi=2),
        # a caller that may not allocate (capture, serving): the allocation-free C entry on a small odd-sized cavity
        _cavity("small_noalloc_mixed", 31, 17, "NC", 16, "vanLeer", 0.05, "mixed", "noalloc", 4),
        # bench.py --workload cavity_64, in both precisions
        _cavity("cavity64_gh24_fp64", 64, 64, "GH", 24, "vanLeer", 0.075, "fp64", "graph", 10),
        _cavity("cavity64_gh24_mixed", 64, 64, "GH", 24, "vanLeer", 0.075, "mixed", "graph", 10),
        # ragged, skewed, non-axis-aligned cells on four blocks with the third limiter: a body-fitted grid
        _cavity("bent_ragged_minmod_fp64", 97, 61, "NC", 24, "minmod", 0.3, "fp64", "plan", 5, nbi=2, nbj=2, bend=0.06),
        # the reference's own call sequence, one launch per reference kernel and block, host readbacks included
        _cavity("per_kernel_64_weno_fp64", 64, 64, "NC", 24, "WENO5", 0.075, "fp64", "one_step", 2),
        # bench.py --workload cavity_2x2 (four blocks of 128 x 128 cells), in both precisions
        _cavity("cavity_2x2x128_weno_fp64", 256, 256, "NC", 32, "WENO5", 0.01, "fp64", "graph", 4, nbi=2, nbj=2),
        _cavity("cavity_2x2x128_weno_mixed", 256, 256, "NC", 32, "WENO5", 0.01, "mixed", "graph", 4, nbi=2, nbj=2),
        # independent uneven cases in one plan: the metric's configuration, 16 of its kind
        dict(name="batch16_weno_fp64", kind="batch", ncases=16, draw_seed=20261202, method="WENO5", CFL=0.8,
             precision="fp64", entry="graph", steps=3),
        dict(name="batch16_weno_mixed", kind="batch", ncases=16, draw_seed=20261202, method="WENO5", CFL=0.8,
             precision="mixed", entry="graph", steps=4),
        # bench.py --workload channel: inflow, extrapolation, adsorbing and diffuse walls, 8 blocks of uneven width
        dict(name="channel_adsorbing_fp64", kind="channel", widths="128,96,192,64,160,128,96,160", height=256, nv=40,
             method="WENO5", Kn=0.05, precision="fp64", entry="graph", steps=2),
        # bench.py --workload cavity_512: the largest single case
        _cavity("cavity512_nc48_weno_mixed", 512, 512, "NC", 48, "WENO5", 0.075, "mixed", "graph", 3),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    """A case between the smallest and the largest listed one: any entry, precision, limiter, velocity set and grid."""
    largest = max(work(c)["bytes"] for c in listed())
    while True:
        case = _draw_any(rng)
        if work(case)["bytes"] <= largest and _updates(case) <= MAX_UPDATES:
            return case


def _draw_any(rng):
    kind = rng.choices(("cavity", "batch", "channel"), (8, 2, 2))[0]
    precision = rng.choice(("fp64", "mixed"))
    entry = rng.choice(("plan", "graph"))
    method = rng.choices(METHODS, (3, 5, 1))[0]
    steps = rng.randint(1, 6)
    Kn = round(_log(rng, 1e-3, 1.0), 6)
    if kind == "batch":
        return dict(kind="batch", ncases=rng.randint(2, 10), draw_seed=rng.randrange(1 << 30), method=method, CFL=0.8,
                    precision=precision, entry=entry, steps=min(steps, 3))
    if kind == "channel":
        widths = [int(_log(rng, 8, 96)) for _ in range(rng.randint(1, 6))]
        return dict(kind="channel", widths=",".join(map(str, widths)), height=int(_log(rng, 8, 160)),
                    nv=rng.choice(BATCH_GRIDS), method=method, Kn=Kn, precision=precision, entry=entry, steps=steps)
    ni, nj = int(_log(rng, 8, 320)), int(_log(rng, 8, 320))
    vel, nv = rng.choice((("GH", rng.randint(8, 28)), ("NC", rng.choice((8, 12, 16, 24, 32, 40, 48)))))
    nbi, nbj = rng.randint(1, 1 + (ni >= 16)), rng.randint(1, 1 + (nj >= 16))
    if ni * nj * nv * nv <= 3e6 and rng.random() < 0.4:
        entry, nbi, nbj = rng.choice((("noalloc", nbi, nbj), ("one_step", 1, 1)))
    return _cavity(None, ni, nj, vel, nv, method, Kn, "fp64" if entry == "one_step" else precision, entry, steps,
                   nbi, nbj, rng.choice((0.0, 0.0, 0.05)))


def _batch_members(case):
    """Side, velocity grid, Kn, lid and wall temperature of each case of a batch (cases.cfg4_batch's ranges)."""
    r = np.random.default_rng(case["draw_seed"])
    return [dict(side=int(r.choice(BATCH_SIDES)), nv=int(r.choice(BATCH_GRIDS)), Kn=float(10.0 ** r.uniform(-3.0, 0.0)),
                 lid=float(r.uniform(0.05, 0.3)), wall_T=float(r.uniform(0.8, 1.2))) for _ in range(case["ncases"])]


def _axis_count(vel, nv):
    return nv if vel == "GH" else nv // 4 * 4 + 1


def _updates(case):
    if case["kind"] == "batch":
        return sum(m["side"] ** 2 * _axis_count("NC", m["nv"]) ** 2 for m in _batch_members(case))
    if case["kind"] == "channel":
        return sum(map(int, case["widths"].split(","))) * case["height"] * _axis_count("NC", case["nv"]) ** 2
    return case["ni"] * case["nj"] * _axis_count(case["vel"], case["nv"]) ** 2


def work(case):
    """Each pass reads and writes the (g, h) pair of every cell and velocity once per step, and loads the initial
    state once; the operations are one interface flux per face and velocity and one update, of a few hundred each."""
    upd = _updates(case)
    pair = 8 if case["precision"] == "mixed" else 16
    per = 400 if case["method"] == "WENO5" else 300
    return {"bytes": 2.0 * pair * upd * (case["steps"] + 1), "flops": float(per) * upd * case["steps"]}


# ------------------------------------------------------------------ inputs --
class Flow:
    """A smooth initial flow (rho, U, V, T) at (x, y): six random Fourier modes per field, drawn from the seed."""
    AMPLITUDE = (0.02, 0.02, 0.02, 0.01)

    def __init__(self, seed, U0=0.0, scale=1.0):
        r = np.random.default_rng([20261202, seed])
        self.k = r.integers(1, 9, (4, 6, 2)) * math.pi / scale
        self.phase = r.uniform(0, 2 * math.pi, (4, 6))
        self.amp = np.array(self.AMPLITUDE)[:, None] * r.uniform(0.3, 1.0, (4, 6)) / 3.0
        self.base = (1.0, U0, 0.0, 1.0)

    def at(self, x, y):
        out = np.empty(x.shape + (4,))
        for q in range(4):
            f = np.full(x.shape, self.base[q])
            for a, k, p in zip(self.amp[q], self.k[q], self.phase[q]):
                f += a * np.cos(k[0] * x + k[1] * y + p)
            out[..., q] = f
        return out


def _centres(v):
    return 0.25 * (v[:-1, :-1] + v[1:, :-1] + v[:-1, 1:] + v[1:, 1:])


def _domains(case, seed):
    """The independent domains of a case: what both the simulation and ``exact`` are built from."""
    if case["kind"] == "batch":
        return [dict(ni=m["side"], nj=m["side"], nbi=1, nbj=1, vel="NC", nv=m["nv"], Kn=m["Kn"], lid=m["lid"],
                     wall_T=m["wall_T"], method=case["method"], CFL=case["CFL"], bend=0.0, widths=None, length=1.0,
                     flow=Flow(64 * seed + k)) for k, m in enumerate(_batch_members(case))]
    if case["kind"] == "channel":
        w = [int(x) for x in case["widths"].split(",")]
        return [dict(ni=sum(w), nj=case["height"], widths=w, vel="NC", nv=case["nv"], Kn=case["Kn"], lid=0.0,
                     wall_T=1.0, method=case["method"], CFL=0.8, bend=0.0, length=4.0, flow=Flow(64 * seed, 0.5, 2.0))]
    return [dict(case, lid=0.15, wall_T=1.0, widths=None, length=1.0, flow=Flow(64 * seed))]


def _gdata(d):
    if d["widths"]:
        g = wl.cfg5_channel(d["widths"], d["nj"], d["nv"], d["Kn"], d["method"], length=d["length"])
    else:
        g = wl.cavity(d["ni"], (d["vel"], d["nv"]), d["method"], d["Kn"], lid=d["lid"], wall_T=d["wall_T"],
                      nb=(d["nbi"], d["nbj"]), CFL=d["CFL"], n_cells_j=d["nj"])
        if d["bend"]:
            wl.curvilinear(g, d["bend"])
    for b in g.blocks:
        b.init_macro = d["flow"].at(_centres(b.x), _centres(b.y))
    return g


class _View:
    """A block's device array for torch, without a copy; holds the array while a tensor of it lives."""

    def __init__(self, arr):
        self.arr = arr
        self.__cuda_array_interface__ = dict(shape=arr.shape, typestr=arr.dtype.str, data=(arr.ptr, False), version=2)


def _tensor(arr):
    return torch.as_tensor(_View(arr), device="cuda")


def prepare(case, seed):
    sims = [UGKSim(_gdata(d)) for d in _domains(case, seed)]
    mixed, entry = case["precision"] == "mixed", case["entry"]
    s = dict(sims=sims, entry=entry, steps=case["steps"])
    if entry == "noalloc":
        blocks, bufs, bcs, handles, _, dts = plan_inputs(sims, case["precision"])
        s["call"] = (handles, bufs, bcs, len(blocks), L.UGKS_MIXED if mixed else L.UGKS_FP64)
        s["dt"] = L.DeviceArray.from_host(np.frombuffer(bytes(dts[0]), dtype=np.uint8))
    elif entry in ("plan", "graph"):
        s["plan"] = StepPlan(sims, case["precision"], graph=entry == "graph")
    s["load"], s["out"] = [], []
    for b in (b for sim in sims for b in sim.blocks):
        f = b.f32_D if mixed else b.f_D
        held = [f, b.macro_D]
        result = dict(f=_tensor(f), macro=_tensor(b.macro_D), Q=_tensor(b.Q_D), wall_fluxes=_tensor(b.wall_fluxes_D))
        if any(x.type_of_BC == bcd.ADSORBING for x in b.bc_list):
            held.append(b.wall_cover_D)
            result["wall_cover"] = _tensor(b.wall_cover_D)
        for arr in held:
            start = L.DeviceArray(arr.shape, arr.dtype)
            start.copy_from(arr)
            s["load"].append((arr, start))
        s["out"].append(result)
    L.synchronize()
    return s


def run(state):
    for arr, start in state["load"]:
        arr.copy_from(start)
    entry, steps = state["entry"], state["steps"]
    if entry == "one_step":
        for _ in range(steps):
            state["sims"][0].one_step(True)
    elif entry == "noalloc":
        L.check(L.load().ugks_step_run_noalloc(*state["call"], ctypes.c_void_p(state["dt"].ptr), steps, None))
    else:
        state["plan"].run(steps)
    return state["out"]


# ------------------------------------------------- the step in 64 bits --
def _sig12(x):
    return float("%.12g" % x)


def _velocities(vel, nv):
    """Node pairs and weights: Gauss-Hermite with the Gaussian divided out, or composite Boole whose end weight is
    14/15 (ugks_data.py:404-417)."""
    if vel == "GH":
        x, w = np.polynomial.hermite.hermgauss(nv)
        w = w * np.exp(x ** 2)
    else:
        n = _axis_count("NC", nv)
        h = 12.0 / (n - 1)
        x = -6.0 + h * np.arange(n)
        k = np.arange(n)
        w = np.where(k % 4 == 0, 28 / 45, np.where(k % 4 == 2, 24 / 45, 64 / 45))
        w[0] = w[-1] = 14 / 15
        w = w * h
    return np.repeat(x, len(x)), np.tile(x, len(x)), np.outer(w, w).ravel()


def _slope(c, un, dist, rd1, method):
    """Upwind face value and slope of one component from the cells along the normal (iFace, clUGKS.c:110-199);
    dist, rd1: the upwind cell's distance to the face and to the cell behind it, (below, above)."""
    up = un > 0
    pick = lambda a, b: torch.where(up, a, b)  # noqa: E731
    d = pick(dist[0], dist[1])
    n = len(c)
    if method == "WENO5":
        s = [pick(c[k], c[n - 1 - k]) for k in range(5)]
        eps = 1e-16
        b0 = 13 / 12 * (s[0] - 2 * s[1] + s[2]) ** 2 + 0.25 * (s[0] - 4 * s[1] + 3 * s[2]) ** 2
        b1 = 13 / 12 * (s[1] - 2 * s[2] + s[3]) ** 2 + 0.25 * (s[1] - s[3]) ** 2
        b2 = 13 / 12 * (s[2] - 2 * s[3] + s[4]) ** 2 + 0.25 * (3 * s[2] - 4 * s[3] + s[4]) ** 2
        a0, a1, a2 = 0.1 / (eps + b0) ** 2, 0.6 / (eps + b1) ** 2, 0.3 / (eps + b2) ** 2
        f0 = (2 * s[0] - 7 * s[1] + 11 * s[2]) / 6 - s[2]
        f1 = (-s[1] + 5 * s[2] + 2 * s[3]) / 6 - s[2]
        f2 = (2 * s[2] + 5 * s[3] - s[4]) / 6 - s[2]
        sg, mid = (a0 * f0 + a1 * f1 + a2 * f2) / (a0 + a1 + a2) / d, s[2]
    else:
        s = [pick(c[k], c[n - 1 - k]) for k in range(3)]
        mid = s[1]
        if method == "vanLeer":
            r = pick(rd1[0], rd1[1])
            p, q = (s[1] - s[0]) / r, (s[2] - s[1]) / r
            sg = (torch.sign(p) + torch.sign(q)) * p.abs() * q.abs() / (p.abs() + q.abs() + 1e-16)
        else:
            p, q = s[2] - s[1], s[1] - s[0]
            mm = torch.where((p * q > 0) & (p.abs() < q.abs()), p, torch.where((p * q > 0) & (q.abs() < p.abs()), q,
                             torch.where(p == q, p, torch.zeros_like(p))))
            sg = 0.5 * mm / d
    return mid + sg * d, sg


class _Exact:
    """One domain stepped in 64 bits (ugks_sim.py:407-501 over clUGKS.c's kernels), whole, in chunks of velocities."""

    def __init__(self, d, dev):
        self.d, self.dev = d, dev
        T = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=dev)  # noqa: E731
        self.ni, self.nj, self.method = d["ni"], d["nj"], d["method"]
        self.G = G = 3 if self.method == "WENO5" else 2
        u, v, w = _velocities(d["vel"], d["nv"])
        self.nv = len(u)
        self.u, self.v, self.w = T(u), T(v), T(w)
        self.umax, self.vmax = _sig12(abs(u.max())), _sig12(abs(v.max()))
        self.Pr, self.gam, self.K, self.Kn, self.CFL = _sig12(2 / 3), _sig12(5 / 3), 1.0, d["Kn"], d["CFL"]
        x, y = np.meshgrid(d["length"] * np.arange(self.ni + 1) / self.ni, np.arange(self.nj + 1) / self.nj, indexing="ij")
        if d["bend"]:
            bump = d["bend"] * np.sin(np.pi * x) * np.sin(np.pi * y)
            x, y = x + bump * np.sin(2 * np.pi * y), y - bump * np.sin(2 * np.pi * x)
        m = d["flow"].at(_centres(x), _centres(y))
        self._geometry(x, y, T)
        cells = self.ni * self.nj
        self.chunk = max(1, min(self.nv, int(2.5e7 // cells)))
        self.macro = T(np.concatenate([m[..., :3], 1 / m[..., 3:]], -1))
        shape = (self.ni + 2 * G, self.nj + 2 * G, self.nv)
        self.g, self.h = (torch.zeros(shape, dtype=torch.float64, device=dev) for _ in range(2))
        self.Q = torch.zeros(self.ni, self.nj, 2, dtype=torch.float64, device=dev)
        for c in self._chunks():
            self.inner(self.g)[..., c], self.inner(self.h)[..., c] = self._equilibrium(self.macro, self.Q, c)
        s = self._cell_sums(lambda g, h, u, v: (g, u * g, v * g, 0.5 * ((u * u + v * v) * g + h)))
        self.macro = self._primary(torch.stack(s, -1))
        self.Q = self._heat(self.macro)
        wl_ = max(self.ni, self.nj)
        self.cover, self.wall_fluxes = (torch.zeros(wl_, 4, n, dtype=torch.float64, device=dev) for n in (4, 8))
        # per side N, E, S, W: kind, and the wall's (rho, U, V, 1/T)
        wall = lambda kind, U=0.0: (kind, (1.0, _sig12(U), 0.0, 1 / _sig12(d["wall_T"])))  # noqa: E731
        self.sides = ([wall("diffuse"), ("extrapolate", None), wall("adsorbing"), wall("inflow")] if d["widths"] else
                      [wall("diffuse", d["lid"])] + [wall("diffuse")] * 3)
        self._ghosts()
        self.dt = self._time_step()

    def _geometry(self, x, y, T):
        """cellGeom on the grid with linearly continued ghost vertices (clGhostRoutines.c:302-398)."""
        G, ext = self.G, []
        for a in (x, y):
            for ax in (0, 1):
                first, second = np.take(a, [0], ax), np.take(a, [1], ax)
                last, before = np.take(a, [-1], ax), np.take(a, [-2], ax)
                lo = [first + k * (first - second) for k in range(G, 0, -1)]
                hi = [last + k * (last - before) for k in range(1, G + 1)]
                a = np.concatenate(lo + [a] + hi, ax)
            ext.append(a)
        X, Y = ext
        A, B, C, D = ((X[i, j], Y[i, j]) for i, j in (((slice(1, None)), (slice(None, -1))), ((slice(1, None)), (slice(1, None))),
                                                      ((slice(None, -1)), (slice(1, None))), ((slice(None, -1)), (slice(None, -1)))))
        cross = lambda p, q: p[0] * q[1] - q[0] * p[1]  # noqa: E731
        loop = ((A, B), (B, C), (C, D), (D, A))
        area = 0.5 * sum(cross(p, q) for p, q in loop)
        cx = sum((p[0] + q[0]) * cross(p, q) for p, q in loop) / (6 * area)
        cy = sum((p[1] + q[1]) * cross(p, q) for p, q in loop) / (6 * area)
        inner = (slice(G, -G), slice(G, -G))
        self.area = T(area[inner])
        pts = [(p[0][inner], p[1][inner]) for p in (A, B, C, D)]
        span = lambda q: np.max([np.abs(pts[i][q] - pts[j][q]) for i in range(4) for j in range(i)], 0)  # noqa: E731
        self.dx, self.dy = T(span(0)), T(span(1))
        self.faces = []
        for ax, tail, head in ((1, D, A), (0, C, D)):          # S: normal of D -> A, W: of C -> D, turned left
            tx, ty = head[0] - tail[0], head[1] - tail[1]
            ln = np.hypot(tx, ty)
            mx, my = 0.5 * (head[0] + tail[0]), 0.5 * (head[1] + tail[1])
            n = self.ni if ax == 0 else self.nj
            along = slice(G, -G)
            f = lambda a, k=0: np.moveaxis(a, ax, 0)[G + k:G + k + n + 1, along]  # noqa: E731
            gap = lambda k: np.hypot(f(mx) - f(cx, k), f(my) - f(cy, k))  # noqa: E731
            back = lambda k, j: np.hypot(f(cx, k) - f(cx, j), f(cy, k) - f(cy, j))  # noqa: E731
            self.faces.append(dict(ax=ax, n=n, nx=T(f(-ty / ln)), ny=T(f(tx / ln)), len=T(f(ln)), dist=(T(gap(-1)), T(gap(0))),
                                   rd1=(T(back(-1, -2)), T(back(0, 1)))))

    # -- pieces ------------------------------------------------------------
    def inner(self, a):
        return a[self.G:-self.G, self.G:-self.G]

    def _chunks(self):
        return [slice(k, min(k + self.chunk, self.nv)) for k in range(0, self.nv, self.chunk)]

    def _cell_sums(self, terms, where=None):
        g, h = where or (self.inner(self.g), self.inner(self.h))
        acc = None
        for c in self._chunks():
            t = [x.sum(-1) for x in terms(g[..., c], h[..., c], self.u[c], self.v[c])]
            acc = t if acc is None else [a + b for a, b in zip(acc, t)]
        return acc

    def _heat(self, p):
        U, V = p[..., 1:2], p[..., 2:3]
        def terms(g, h, u, v):
            t = ((u - U) ** 2 + (v - V) ** 2) * g + h / self.K
            return 0.5 * (u - U) * t, 0.5 * (v - V) * t
        return torch.stack(self._cell_sums(terms), -1)

    def _primary(self, w):
        r, a, b, e = w.unbind(-1)
        return torch.stack([r, a / r, b / r, 0.5 * r / (self.gam - 1) / (e - 0.5 * (a * a + b * b) / r)], -1)

    def _maxwell(self, p, u, v, w):
        r, U, V, lam = (p[..., k:k + 1] for k in range(4))
        g = w * r * lam / math.pi * torch.exp(-lam * ((u - U) ** 2 + (v - V) ** 2))
        return g, g * self.K / (2 * lam)

    def _shakhov(self, p, Q, u, v, M):
        r, U, V, lam = (p[..., k:k + 1] for k in range(4))
        s = 0.8 * (1 - self.Pr) * lam ** 2 / r * ((u - U) * Q[..., 0:1] + (v - V) * Q[..., 1:2])
        t = 2 * lam * ((u - U) ** 2 + (v - V) ** 2)
        return s * (t - 4) * M[0], s * (t - 2) * M[1]

    def _equilibrium(self, p, Q, c):
        u, v = self.u[c], self.v[c]
        M = self._maxwell(p, u, v, self.w[c])
        S = self._shakhov(p, Q, u, v, M)
        return M[0] + S[0], M[1] + S[1]

    def _tau(self, p):
        return self.Kn / p[..., 0] * p[..., 3] ** (1 - 0.81)

    def _time_step(self):
        U, V, lam = self.macro[..., 1].abs(), self.macro[..., 2].abs(), self.macro[..., 3]
        sos = torch.sqrt(0.5 * self.gam / lam)
        scale = (math.erf(10 * (self.Kn - 1e-3)) + 1) / 2
        def speed(a, top):
            a = a + sos
            lo, hi = a.clamp(max=top), a.clamp(min=top)
            return scale * (hi - lo) + lo
        return self.CFL / float(((self.dx * speed(U, self.umax) + self.dy * speed(V, self.vmax)) / self.area).max())

    def _ghosts(self):
        """updateBC of the four sides (ugks_block.py:621-665)."""
        G, n = self.G, (self.ni, self.nj)
        for side, (kind, wall) in enumerate(self.sides):
            ax, high = (1, 0)[side % 2], side < 2
            along = slice(G, G + n[1 - ax])
            e0, inward = (G + n[ax] - 1, -1) if high else (G, 1)
            for name in ("g", "h"):
                a = getattr(self, name).movedim(ax, 0)
                for m in range(1, G + 1):
                    edge, second = a[e0, along], a[e0 + inward, along]
                    if kind == "extrapolate":
                        a[e0 - inward * m, along] = edge
                    elif kind != "inflow":
                        a[e0 - inward * m, along] = edge + m * (edge - second)
            if kind == "inflow":
                p, q = (t.movedim(ax, 0)[-1 if high else 0].clone() for t in (self.macro, self.Q))
                p[..., 0], p[..., 3] = wall[0], wall[3]
                eq = self._equilibrium(p, q, slice(None))
                for m in range(1, G + 1):
                    self.g.movedim(ax, 0)[e0 - inward * m, along], self.h.movedim(ax, 0)[e0 - inward * m, along] = eq

    # -- faces ---------------------------------------------------------------
    def _stencil(self, f, a, c, only=None):
        """The cells along the normal of every face of one direction (face axis first), own cell at index R."""
        R, G = (3 if self.method == "WENO5" else 2), self.G
        a = a.movedim(f["ax"], 0)[:, G:-G, c]
        lo, hi = (G, G + f["n"] + 1) if only is None else (G + only, G + only + 1)
        return [a[lo + k:hi + k] for k in range(-R, R)]

    def _face_values(self, f, c, only=None):
        """Face-frame velocities, face values and slopes of g and h, and the cells below and above."""
        sel = slice(None) if only is None else slice(only, only + 1)
        e = lambda t: t[sel].unsqueeze(-1)  # noqa: E731
        nx, ny, u, v = e(f["nx"]), e(f["ny"]), self.u[c], self.v[c]
        un, ut = u * nx + v * ny, v * nx - u * ny
        dist, rd1 = [e(t) for t in f["dist"]], [e(t) for t in f["rd1"]]
        cg, ch = self._stencil(f, self.g, c, only), self._stencil(f, self.h, c, only)
        R = len(cg) // 2
        return (un, ut, *_slope(cg, un, dist, rd1, self.method), *_slope(ch, un, dist, rd1, self.method),
                cg[R - 1], ch[R - 1], cg[R], ch[R])

    def _micro_slope(self, p, s):
        K = self.K
        r, U, V, lam = p.unbind(-1)
        s0, s1, s2, s3 = s.unbind(-1)
        a3 = 4 * lam ** 2 / (K + 2) / r * (2 * s3 - 2 * U * s1 - 2 * V * s2 + s0 * (U * U + V * V - 0.5 * (K + 2) / lam))
        a2 = 2 * lam / r * (s2 - V * s0) - V * a3
        a1 = 2 * lam / r * (s1 - U * s0) - U * a3
        return torch.stack([s0 / r - U * a1 - V * a2 - 0.5 * (U * U + V * V + 0.5 * (K + 2) / lam) * a3, a1, a2, a3], -1)

    def _half_moments(self, p):
        _, U, V, lam = p.unbind(-1)
        ex = 0.5 * torch.exp(-lam * U * U) / torch.sqrt(math.pi * lam)
        left, right = [0.5 * torch.erfc(-torch.sqrt(lam) * U)], [0.5 * torch.erfc(torch.sqrt(lam) * U)]
        left.append(U * left[0] + ex)
        right.append(U * right[0] - ex)
        tang = [torch.ones_like(U), V]
        for i in range(2, 7):
            left.append(U * left[-1] + 0.5 * (i - 1) * left[-2] / lam)
            right.append(U * right[-1] + 0.5 * (i - 1) * right[-2] / lam)
            tang.append(V * tang[-1] + 0.5 * (i - 1) * tang[-2] / lam)
        K = self.K
        return left, right, tang, [torch.ones_like(U), 0.5 * K / lam, (K * K + 2 * K) / (4 * lam ** 2)]

    def _flux(self, f, dt):
        """UGKS_flux of one direction (ugks_block.py:1062-1257): per-velocity and macro fluxes, face axis first."""
        ax, n = f["ax"], f["n"]
        high, low = (1, 3) if ax == 0 else (0, 2)              # side numbers of the last and the first face
        walls = [(k, s) for k, s in ((n, high), (0, low)) if self.sides[s][0] in ("diffuse", "adsorbing")]
        psi = lambda g, h, a, b: torch.stack([t.sum(-1) for t in (g, a * g, b * g, 0.5 * ((a * a + b * b) * g + h))], -1)  # noqa: E731
        W = WL = WR = 0
        for c in self._chunks():
            un, ut, fg, _, fh, _, lg, lh, rg, rh = self._face_values(f, c)
            W, WL, WR = W + psi(fg, fh, un, ut), WL + psi(lg, lh, un, ut), WR + psi(rg, rh, un, ut)
        p = self._primary(W)
        aL = self._micro_slope(p, (W - WL) / f["dist"][0].unsqueeze(-1))
        aR = self._micro_slope(p, (WR - W) / f["dist"][1].unsqueeze(-1))
        ml, mr, mt, mx = self._half_moments(p)
        full = [a + b for a, b in zip(ml, mr)]
        def uv(mu, a, b, d=0):
            return torch.stack([mu[a] * mt[b] * mx[d], mu[a + 1] * mt[b] * mx[d], mu[a] * mt[b + 1] * mx[d],
                                0.5 * (mu[a + 2] * mt[b] * mx[d] + mu[a] * mt[b + 2] * mx[d] + mu[a] * mt[b] * mx[d + 1])], -1)
        def au(s, mu, a):
            s0, s1, s2, s3 = (s[..., k:k + 1] for k in range(4))
            return s0 * uv(mu, a, 0) + s1 * uv(mu, a + 1, 0) + s2 * uv(mu, a, 1) + 0.5 * s3 * (uv(mu, a + 2, 0) + uv(mu, a, 2) + uv(mu, a, 0, 1))
        rho = p[..., 0:1]
        aT = self._micro_slope(p, -rho * (au(aL, ml, 1) + au(aR, mr, 1)))
        tau = self._tau(p)
        e = torch.exp(-dt / tau)
        m3 = tau * (1 - e)
        m4 = -tau * dt * e + tau * m3
        m0 = dt - m3
        m1, m2 = -tau * m0 + m4, dt * dt / 2 - tau * m0
        x = lambda t: t.unsqueeze(-1)  # noqa: E731
        macro = rho * (x(m0) * uv(full, 1, 0) + x(m1) * (au(aL, ml, 2) + au(aR, mr, 2)) + x(m2) * au(aT, full, 1))
        Q = 0
        for c in self._chunks():
            un, ut, fg, _, fh, _ = self._face_values(f, c)[:6]
            cu, cv = un - p[..., 1:2], ut - p[..., 2:3]
            t = (cu * cu + cv * cv) * fg + fh / self.K
            Q = Q + torch.stack([(0.5 * cu * t).sum(-1), (0.5 * cv * t).sum(-1)], -1)
        wall_values = {k: self._wall(f, k, s, dt) for k, s in walls}
        ln, nx, ny = f["len"], f["nx"], f["ny"]
        out_g = torch.empty((n + 1, nx.shape[1], self.nv), dtype=torch.float64, device=self.dev)
        out_h = torch.empty_like(out_g)
        for c in self._chunks():
            un, ut, fg, sg, fh, sh = self._face_values(f, c)[:6]
            M = self._maxwell(p, un, ut, self.w[c])
            S = self._shakhov(p, Q, un, ut, M)
            uu, up = un * un + ut * ut, un > 0
            a = [torch.where(up, x(aL[..., k]), x(aR[..., k])) for k in range(4)]
            poly = lambda s, s0, s1: s[0] * s0 + s[1] * un * s0 + s[2] * ut * s0 + 0.5 * s[3] * (uu * s0 + s1)  # noqa: E731
            aTk = [x(aT[..., k]) for k in range(4)]
            kin_g, kin_h = x(m0) * un * S[0] + x(m3) * un * fg - x(m4) * un ** 2 * sg, x(m0) * un * S[1] + x(m3) * un * fh - x(m4) * un ** 2 * sh
            macro = macro + psi(kin_g, kin_h, un, ut)
            out_g[..., c] = x(ln) * (x(m0) * un * M[0] + x(m1) * un ** 2 * poly(a, M[0], M[1]) + x(m2) * un * poly(aTk, M[0], M[1]) + kin_g)
            xi = x(mx[2]) * M[0]
            out_h[..., c] = x(ln) * (x(m0) * un * M[1] + x(m1) * un ** 2 * poly(a, M[1], xi) + x(m2) * un * poly(aTk, M[1], xi) + kin_h)
        macro = x(ln) * torch.stack([macro[..., 0], nx * macro[..., 1] - ny * macro[..., 2],
                                     ny * macro[..., 1] + nx * macro[..., 2], macro[..., 3]], -1)
        for k, (g, h, mac) in wall_values.items():
            out_g[k], out_h[k], macro[k] = g, h, mac
        return out_g, out_h, macro

    def _wall(self, f, k, side, dt):
        """A wall's faces: re-emission, wallFlux and wallMassEnergyFluxes (clUGKS.c:776-1147, clAdsorb.c:253-975)."""
        un, ut, g, _, h, _ = (t[0] for t in self._face_values(f, slice(None), k)[:6])
        rot = -1 if side < 2 else 1
        kind, (rho, U, V, lam) = self.sides[side]
        nx, ny, ln = f["nx"][k].unsqueeze(-1), f["ny"][k].unsqueeze(-1), f["len"][k].unsqueeze(-1)
        one = torch.ones_like(nx)
        wall = torch.cat([rho * one, U * nx + V * ny, V * nx - U * ny, lam * one], -1)
        leaves = rot * un > 0
        M = self._maxwell(wall, un, ut, self.w)
        n = len(nx)
        if kind == "diffuse":
            ratio = (torch.where(leaves, 0.0, un * g).sum(-1) / -torch.where(leaves, un * M[0], 0.0).sum(-1)).unsqueeze(-1)
            eg, eh = ratio * M[0], ratio * M[1]
        else:
            gf, veq = 0.3, float("%g" % (0.3 / 0.31))
            theta = self.cover[:n, side, 0]
            total = torch.where(leaves, 0.0, -rot * un * g)
            ads = total * gf * (1 - theta.unsqueeze(-1))
            ads = torch.where(torch.sign(total) * ads > torch.sign(total) * total, total, ads)
            r0, a0, hit = (total - ads).sum(-1), ads.sum(-1), total.sum(-1)
            dth = dt * a0
            full = dth > 1 - theta
            dth = torch.where(full, 1 - theta, dth)
            a1 = torch.where(full, dth / dt, a0)
            des = gf * (1 / veq - 1) * hit * theta
            dth = dth - dt * des
            des = torch.where(theta + dth < 0, theta / dt, des)
            refl = r0 + a0 - a1
            self.cover[:n, side] = torch.stack([theta + dth, refl, a1, des], -1)
            ratio = (refl / torch.where(leaves, rot * un * M[0], 0.0).sum(-1)).unsqueeze(-1)
            wall[..., 0] = 2 * des * torch.sqrt(math.pi * wall[..., 3])
            D = self._maxwell(wall, un, ut, self.w)
            eg, eh = ratio * M[0] + D[0], ratio * M[1] + D[1]
        g, h = torch.where(leaves, eg, g), torch.where(leaves, eh, h)
        Fg, Fh = un * g * ln * dt, un * h * ln * dt
        t = [Fg, un * Fg, ut * Fg, 0.5 * ((un * un + ut * ut) * Fg + Fh)]
        m = [a.sum(-1) for a in t]
        for q in range(4):
            self.wall_fluxes[:n, side, 2 * q] = -rot * torch.where(leaves, 0.0, t[q]).sum(-1)
            self.wall_fluxes[:n, side, 2 * q + 1] = rot * torch.where(leaves, t[q], 0.0).sum(-1)
        nx, ny = nx[..., 0], ny[..., 0]
        return Fg, Fh, torch.stack([m[0], nx * m[1] - ny * m[2], ny * m[1] + nx * m[2], m[3]], -1)

    def step(self):
        dt, old = self.dt, self.macro
        self.Q = self._heat(old)
        net_g = net_h = net = 0
        for f in self.faces:
            g, h, mac = self._flux(f, dt)
            d = lambda t: (t[:-1] - t[1:]).movedim(0, f["ax"])  # noqa: E731
            net_g, net_h, net = net_g + d(g), net_h + d(h), net + d(mac)
            del g, h
        r, U, V, lam = old.unbind(-1)
        w = torch.stack([r, r * U, r * V, 0.5 * r / lam / (self.gam - 1) + 0.5 * r * (U * U + V * V)], -1)
        new = self._primary(w + net / self.area.unsqueeze(-1))
        x = lambda t: t.unsqueeze(-1)  # noqa: E731
        a, b, A = x(0.5 * dt / self._tau(new)), x(0.5 * dt / self._tau(old)), x(self.area)
        for c in self._chunks():
            eo, en = self._equilibrium(old, self.Q, c), self._equilibrium(new, self.Q, c)
            for arr, nt, k in ((self.inner(self.g), net_g, 0), (self.inner(self.h), net_h, 1)):
                arr[..., c] = (arr[..., c] + nt[..., c] / A + a * en[k] + b * (eo[k] - arr[..., c])) / (1 + a)
        self.macro = new
        self.dt = self._time_step()
        self._ghosts()

    def blocks(self):
        """The state laid out block by block as the simulation holds it (corner ghost cells are never filled)."""
        d, G = self.d, self.G
        def cuts(n, nb):
            out, at = [], 0
            for k in range(nb):
                m = (n - at) // (nb - k)
                out.append((at, at + m))
                at += m
            return out
        if d["widths"]:
            edge = np.cumsum([0] + d["widths"])
            si, sj = list(zip(edge[:-1], edge[1:])), [(0, self.nj)]
        else:
            si, sj = cuts(self.ni, d["nbi"]), cuts(self.nj, d["nbj"])
        out = []
        for i, (i0, i1) in enumerate(si):
            for j, (j0, j1) in enumerate(sj):
                f = torch.stack([t[i0:i1 + 2 * G, j0:j1 + 2 * G] for t in (self.g, self.h)], -1)
                for a in (slice(0, G), slice(-G, None)):
                    for b in (slice(0, G), slice(-G, None)):
                        f[a, b] = 0
                length = max(i1 - i0, j1 - j0)
                # a side inside the domain is a join: it has no wall state
                at = {0: j1 == self.nj, 1: i1 == self.ni, 2: j0 == 0, 3: i0 == 0}
                def side_state(t):
                    o = torch.zeros(length, 4, t.shape[-1], dtype=torch.float64, device=self.dev)
                    for s in range(4):
                        lo, hi = (i0, i1) if s % 2 == 0 else (j0, j1)
                        if at[s]:
                            o[:hi - lo, s] = t[lo:hi, s]
                    return o
                r = dict(f=f, macro=self.macro[i0:i1, j0:j1], Q=self.Q[i0:i1, j0:j1], wall_fluxes=side_state(self.wall_fluxes))
                if d["widths"]:
                    r["wall_cover"] = side_state(self.cover)
                out.append(r)
        return out


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    out = []
    for d in _domains(case, seed):
        e = _Exact(d, dev)
        for _ in range(case["steps"]):
            e.step()
        out += e.blocks()
    return out
