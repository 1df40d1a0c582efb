"""Performance cases of the CCZ4 engine: what its users have it do, through the public entry points.

A run of the engine is RK3 steps of blocks, of sets of levels and of whole hierarchies, with
the telemetry in between; a host code that adopts it call by call uses the right-hand side on
its own arrays. `listed()` holds one case of each, from a latency-bound 32^3 box to a 192^3
block and a whole Berger-Oliger coarse step; `draw()` gives more of the same ranges.

kind        one pass
step        one SSP-RK3 step of one block held on the device (Level.rk3_step)
matter      the same step stage by stage with matter sources (Level.rk3_stage), as a driver
            whose sources come from another solver runs it
levels      one step of a set of levels of uneven blocks (levels_rk3_step)
hierarchy   one coarse step of a Berger-Oliger hierarchy (Hierarchy.step)
telemetry   constraint norms, CFL and NaN scan of a hierarchy between steps
rhs_host    CCZ4Evolution.computeRHS on host arrays, the drop-in for a host code's own call
rhs_device  gr_ccz4_rhs_device on the caller's device arrays
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

import granite_amd as ga
from granite_amd import hierarchy as hy
from granite_amd import workloads

NG = 4
NV = 22
HALF = 16.0  # half width of a single-puncture domain
NOISY = [1, 2, 3, 4, 5, 6, 13]  # conformal metric and K
PARAMS = dict(kappa1=0.02, kappa2=0.0, eta=2.0, ko_sigma=0.1)
MAX_CELLS = 192 ** 3


# ----------------------------------------------------------------------------------------
# the cases
# ----------------------------------------------------------------------------------------
def _step(nx, ny, nz, data="puncture", precision="fp64", graph=True):
    return dict(kind="step", nx=nx, ny=ny, nz=nz, data=data, precision=precision, graph=graph)


def listed():
    return [
        # the 1-D gauge-wave test box, periodic: the smallest configuration that is run, where
        # launches and latency count; replayed from a graph as every driver does
        dict(_step(32, 32, 32, data="gauge"), name="gauge_wave_32"),
        # a 64^3 puncture block, the size of the published single-puncture runs, launched
        # eagerly, as a caller does that looks at the state between steps
        dict(_step(64, 64, 64, graph=False), name="puncture_64"),
        # a box as regridding cuts it: ragged extents, an odd row length, partial tiles everywhere
        dict(_step(101, 77, 59), name="ragged_101x77x59"),
        # the headline block
        dict(_step(128, 128, 128), name="puncture_128"),
        # the same block in the mixed-precision form
        dict(_step(128, 128, 128, precision="mixed"), name="puncture_128_mixed"),
        # the large noisy block: the state is several times the last-level cache
        dict(_step(192, 192, 192, data="noisy"), name="noisy_192"),
        # evolution with matter: sources written by another solver, stage by stage
        dict(kind="matter", nx=96, ny=96, nz=96, name="matter_96"),
        # one step of four levels of uneven blocks with edges 16..64 (as many blocks as outputs
        # can be returned), launched eagerly, so that changing the level set costs no capture
        dict(kind="levels", blocks=64, layout=20240611, name="uneven_amr_64_blocks"),
        # one coarse step of the four-level binary-puncture hierarchy
        dict(kind="hierarchy", ncells=96, levels=4, precision="fp64", name="binary_hierarchy"),
        # the telemetry line of the same hierarchy, printed every few coarse steps
        dict(kind="telemetry", ncells=96, levels=4, name="binary_telemetry"),
        # the drop-in call of a host code on one of its blocks
        dict(kind="rhs_host", nx=48, ny=48, nz=48, matter=False, name="rhs_host_48"),
        # the right-hand side on device arrays of a caller with its own integrator
        dict(kind="rhs_device", nx=96, ny=96, nz=96, matter=False, name="rhs_device_96"),
    ]


def _extents(rng, lo, hi, cells):
    """Three extents spread over lo..hi on a log scale, near to one another, of at most `cells` cells."""
    while True:
        c = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        n = [max(lo, min(hi, int(round(c * math.exp(rng.uniform(-0.5, 0.5)))))) for _ in range(3)]
        if n[0] * n[1] * n[2] <= cells:
            return n


def draw(rng):
    kind = rng.choices(["step", "matter", "levels", "hierarchy", "telemetry", "rhs_host", "rhs_device"],
                       weights=[50, 8, 10, 10, 6, 6, 10])[0]
    if kind == "step":
        nx, ny, nz = _extents(rng, 12, 192, MAX_CELLS)
        return _step(nx, ny, nz, data=rng.choice(["puncture", "puncture", "noisy", "gauge"]),
                     precision="mixed" if rng.random() < 0.25 else "fp64", graph=rng.random() < 0.7)
    if kind == "levels":
        return dict(kind=kind, blocks=rng.randint(8, 64), layout=rng.randrange(1 << 30))
    if kind in ("hierarchy", "telemetry"):
        case = dict(kind=kind, ncells=2 * rng.randint(16, 48), levels=rng.randint(2, 4))
        if kind == "hierarchy":
            case["precision"] = "mixed" if rng.random() < 0.25 else "fp64"
        return case
    nx, ny, nz = _extents(rng, 12, 64 if kind == "rhs_host" else 128, MAX_CELLS)
    case = dict(kind=kind, nx=nx, ny=ny, nz=nz)
    if kind != "matter":
        case["matter"] = rng.random() < 0.4
    return case


# ----------------------------------------------------------------------------------------
# geometry and inputs
# ----------------------------------------------------------------------------------------
def _box(case):
    """(n, lo, hi) of a single block: cubic cells, the longest edge spanning the domain."""
    n = [case["nx"], case["ny"], case["nz"]]
    if case.get("data") == "gauge":
        return n, [0.0] * 3, [v / n[0] for v in n]  # one wavelength along x
    h = 2 * HALF / max(n)
    return n, [-0.5 * v * h for v in n], [0.5 * v * h for v in n]


def _dx(box):
    n, lo, hi = box
    return [(hi[d] - lo[d]) / float(n[d]) for d in range(3)]


def _geometry(case):
    """[[(n, lo, hi), ...] per level]"""
    kind = case["kind"]
    if kind == "levels":
        return [blocks for _, blocks in workloads.uneven_amr_levels(nblocks=case["blocks"], seed=case["layout"])]
    if kind in ("hierarchy", "telemetry"):
        return hy.binary_puncture_levels(ncells=case["ncells"], max_levels=case["levels"])
    return [[_box(case)]]


def _dt(case):
    """CFL 0.25 on the coarsest level."""
    if case["kind"] in ("hierarchy", "telemetry"):
        return 0.25 * (128.0 / case["ncells"])
    return 0.25 * _dx(_geometry(case)[0][0])[0]


def _punctures(case, seed):
    """Masses and positions, jittered by the seed (and off every cell centre)."""
    r = np.random.default_rng(seed)
    masses, pos = workloads.PUNCTURES if case["kind"] in ("levels", "hierarchy", "telemetry") else ([1.0], [[0.0] * 3])
    return ([m * (1.0 + 0.02 * r.uniform(-1, 1)) for m in masses],
            [[c + 0.05 * r.uniform(-1, 1) for c in p] for p in pos])


class _DeviceView:
    """A block's device state as an array torch can take without a copy; keeps its level alive."""

    def __init__(self, level, index):
        lib = ga.library()
        p = C.c_void_p()
        if lib.gr_level_state(level._h, index, C.byref(p)) != 0:
            raise RuntimeError("no device state")
        self.owner = level
        self.__cuda_array_interface__ = dict(shape=level.blocks[index].array.shape, typestr="<f8",
                                             data=(p.value, False), version=2)


def _tensor(level, index):
    return torch.as_tensor(_DeviceView(level, index), device="cuda")


class _DeviceBlock(ga.GridBlock):
    """A GridBlock without host data, for levels whose state only lives on the device."""

    def __init__(self, level, n, lo, hi):
        super().__init__(0, level, (1, 1, 1), lo, hi, NG)
        self._n = tuple(n)
        self._dx = (self._hi - self._lo) / np.array(self._n, dtype=np.float64)
        nt = [v + 2 * NG for v in n]
        self.array = np.broadcast_to(np.zeros(1), (NV, nt[2], nt[1], nt[0]))


def _make_levels(case, seed):
    """Levels with initial data on the device (finer levels of a hierarchy still empty)."""
    levels = [ga.Level([_DeviceBlock(l, *b) for b in blocks]) for l, blocks in enumerate(_geometry(case))]
    hier = case["kind"] in ("hierarchy", "telemetry")
    data = case.get("data", "puncture")
    r = np.random.default_rng(seed)
    for l, lv in enumerate(levels):
        if hier and l > 0:
            continue
        if data == "gauge":
            lv.init_gauge_wave(0.1 * (1.0 + 0.1 * r.uniform(-1, 1)), 1.0)
        else:
            lv.init_brill_lindquist(*_punctures(case, seed))
        lv.add_noise(seed + 17 * l, 1e-8, NOISY if data == "noisy" else range(NV))
    return levels


def _states(levels):
    return [[_tensor(lv, i) for i in range(len(lv.blocks))] for lv in levels]


def _sources(case, seed):
    """A smooth blob of matter off the centre, with noise: rho, S_i, S_ij, S as device arrays."""
    n, lo, hi = _box(case)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    x = [torch.linspace(-1.0, 1.0, n[d] + 2 * NG, dtype=torch.float64, device="cuda") for d in range(3)]
    r2 = (x[2][:, None, None] - 0.2) ** 2 + (x[1][None, :, None] + 0.3) ** 2 + (x[0][None, None, :] - 0.4) ** 2
    blob = (1e-3 * torch.exp(-4.0 * r2)).reshape(-1, 1)
    make = lambda k: blob * (1.0 + 0.1 * torch.rand(blob.numel(), k, dtype=torch.float64, device="cuda",  # noqa: E731
                                                    generator=gen))
    return [make(1).reshape(-1).contiguous(), 0.1 * make(3), 0.1 * make(6), make(1).reshape(-1).contiguous()]


def _mode(case):
    """The block's boundary: periodic for the gauge wave, else the reference's level-0 semantics."""
    if case.get("data") == "gauge":
        return dict(bc_mode=ga.BC_PERIODIC, pre_fill=ga.BC_PERIODIC)
    return dict(bc_mode=ga.BC_SOMMERFELD, pre_fill=ga.BC_OUTFLOW)


def _precision(case):
    return ga.PREC_MIXED if case.get("precision") == "mixed" else ga.PREC_FP64


def _initial_block(case, seed):
    """The initial state of a single block with ghosts filled, as a device tensor."""
    lv = _make_levels(case, seed)[0]
    lv.fill_ghosts(ga.BC_OUTFLOW)
    return lv, _tensor(lv, 0)


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case, params=ga.CCZ4Params(**PARAMS), dt=_dt(case), engine=ga.Engine.default())
    if kind in ("rhs_host", "rhs_device"):
        lv, u = _initial_block(case, seed)
        src = _sources(case, seed) if case["matter"] else None
        if kind == "rhs_device":
            s.update(u=u.clone(), rhs=torch.zeros_like(u), src=src, geom=lv.blocks[0].geom())
        else:
            n, lo, hi = _box(case)
            grid, rhs = (ga.GridBlock(i, 0, n, lo, hi, NG) for i in range(2))
            grid.array[...] = u.cpu().numpy()
            s.update(grid=grid, rhs=rhs, src=src and [a.cpu().numpy() for a in src],
                     evolution=ga.CCZ4Evolution(s["params"]))
        return s
    s["levels"] = levels = _make_levels(case, seed)
    if kind in ("hierarchy", "telemetry"):
        s["hierarchy"] = H = ga.Hierarchy(levels)
        for l in range(1, len(levels)):
            H.prolongate(l)
        H.fill_ghosts(0)
    if kind == "matter":
        s["src"] = _sources(case, seed)
        torch.cuda.synchronize()
        levels[0].set_sources(0, *[a.data_ptr() for a in s["src"]])
    if kind == "levels":
        s["dts"] = [0.25 * _dx(blocks[0])[0] for blocks in _geometry(case)]
    s["out"] = _states(levels)
    return s


def run(s):
    case, p, dt = s["case"], s["params"], s["dt"]
    kind = case["kind"]
    if kind == "step":
        s["levels"][0].rk3_step(p, dt, _precision(case), use_graph=case["graph"], **_mode(case))
        return s["out"][0][0]
    if kind == "matter":
        lv = s["levels"][0]
        lv.rk3_stage(p, dt, 1, pre_fill=ga.BC_OUTFLOW)
        lv.rk3_stage(p, dt, 2)
        lv.rk3_stage(p, dt, 3)
        return s["out"][0][0]
    if kind == "levels":
        ga.levels_rk3_step(s["levels"], s["dts"], p, pre_fill=ga.BC_OUTFLOW)
        return [u for lv in s["out"] for u in lv]
    if kind == "hierarchy":
        s["hierarchy"].step(p, dt, _precision(case), use_graph=True)
        return [u for lv in s["out"] for u in lv]
    if kind == "telemetry":
        ham, mom, count = s["hierarchy"].constraints_l2()
        out = dict(ham=ham, mom=mom, count=count)
        for l, lv in enumerate(s["levels"]):
            out["cfl%d" % l] = lv.cfl(dt / 2 ** l)
            out["nonfinite%d" % l] = lv.nonfinite()
        return out
    if kind == "rhs_host":
        if s["src"] is None:
            s["evolution"].computeRHSVacuum(s["grid"], s["rhs"])
        else:
            s["evolution"].computeRHS(s["grid"], s["rhs"], *s["src"])
        return s["rhs"].array
    src = [C.c_void_p(a.data_ptr()) for a in s["src"]] if s["src"] else [None] * 4
    eng = s["engine"]
    eng.check(eng.lib.gr_ccz4_rhs_device(eng.handle, C.byref(s["geom"]), C.byref(p.c()), C.c_void_p(s["u"].data_ptr()),
                                         C.c_void_p(s["rhs"].data_ptr()), *src))
    return s["rhs"]


# Floating-point operations per cell that the discretisation asks for: per field and axis the
# centred (7), upwind (10) and dissipation (13) stencils; the second derivatives of ten fields (57);
# then the algebra of the right-hand side, about 1500 (Christoffel symbols, Ricci tensor, contractions).
RHS_FLOPS = NV * 3 * 30 + 10 * 57 + 1500
MONITOR_FLOPS = 7 * (3 * 7 + 57) + 10 * 21 + 1800


def work(case):
    """Every value of the state in and out once (ghosts included); a right-hand side per RK3 stage."""
    geo = _geometry(case)
    whole = [sum(math.prod(v + 2 * NG for v in n) for n, _, _ in lv) for lv in geo]
    inner = [sum(math.prod(n) for n, _, _ in lv) for lv in geo]
    kind = case["kind"]
    if kind in ("rhs_host", "rhs_device"):
        return dict(bytes=8.0 * (NV * (whole[0] + inner[0]) + (11 * inner[0] if case["matter"] else 0)),
                    flops=float(RHS_FLOPS * inner[0]))
    if kind == "telemetry":
        return dict(bytes=8.0 * NV * sum(inner), flops=float(MONITOR_FLOPS * sum(inner)))
    steps = [2 ** l if kind == "hierarchy" else 1 for l in range(len(geo))]
    per_cell = 2 * NV * 8.0 + (11 * 8.0 if kind == "matter" else 0.0)
    return dict(bytes=per_cell * sum(w * k for w, k in zip(whole, steps)),
                flops=3.0 * RHS_FLOPS * sum(c * k for c, k in zip(inner, steps)))


# ----------------------------------------------------------------------------------------
# the same results in plain 64-bit torch
# ----------------------------------------------------------------------------------------
CHI, GXX, AXX, KTR, GHX, THETA, ALPHA, BX = 0, 1, 7, 13, 14, 17, 18, 19
SYM = [[0, 1, 2], [1, 3, 4], [2, 4, 5]]
R3 = range(3)
F_INF = [1.0 if v in (CHI, GXX, GXX + 3, GXX + 5, ALPHA) else 0.0 for v in range(NV)]


def _inner(a):
    return a[..., NG:-NG, NG:-NG, NG:-NG]


def _taps(f, off):
    """f shifted by off = (x, y, z) cells, over the interior."""
    nz, ny, nx = (f.shape[-3 + d] - 2 * NG for d in R3)
    x, y, z = off
    return f[..., NG + z:NG + z + nz, NG + y:NG + y + ny, NG + x:NG + x + nx]


def _unit(d, k):
    return tuple(k if a == d else 0 for a in R3)


def _d1(f, d, h):
    t = lambda k: _taps(f, _unit(d, k))  # noqa: E731
    return (-t(2) + 8 * t(1) - 8 * t(-1) + t(-2)) / (12 * h)


def _d2(f, a, b, h):
    if a == b:
        t = lambda k: _taps(f, _unit(a, k))  # noqa: E731
        return (-t(2) + 16 * t(1) - 30 * t(0) + 16 * t(-1) - t(-2)) / (12 * h[a] * h[a])
    t = lambda i, j: _taps(f, tuple(i if c == a else j if c == b else 0 for c in R3))  # noqa: E731
    return (t(1, 1) - t(1, -1) - t(-1, 1) + t(-1, -1)) / (4 * h[a] * h[b])


def _hessian(f, h):
    up = {(a, b): _d2(f, a, b, h) for a in R3 for b in range(a, 3)}
    return [[up[min(a, b), max(a, b)] for b in R3] for a in R3]


class _Curvature:
    """Inverse metric, Christoffel symbols, the Ricci tensor with its conformal part, A~A~."""

    def __init__(self, u, h, chi):
        self.h, self.chi = h, chi
        m = lambda v: [[_inner(u[v + SYM[a][b]]) for b in R3] for a in R3]  # noqa: E731
        self.g, self.A = g, A = m(GXX), m(AXX)
        self.Gh = Gh = [_inner(u[GHX + a]) for a in R3]
        det = (g[0][0] * (g[1][1] * g[2][2] - g[1][2] ** 2) - g[0][1] * (g[0][1] * g[2][2] - g[1][2] * g[0][2])
               + g[0][2] * (g[0][1] * g[1][2] - g[1][1] * g[0][2])) + 1e-30
        up = {(0, 0): g[1][1] * g[2][2] - g[1][2] ** 2, (0, 1): g[0][2] * g[1][2] - g[0][1] * g[2][2],
              (0, 2): g[0][1] * g[1][2] - g[0][2] * g[1][1], (1, 1): g[0][0] * g[2][2] - g[0][2] ** 2,
              (1, 2): g[0][1] * g[0][2] - g[0][0] * g[1][2], (2, 2): g[0][0] * g[1][1] - g[0][1] ** 2}
        self.gu = gu = [[up[min(a, b), max(a, b)] / det for b in R3] for a in R3]
        dg = [[[_d1(u[GXX + SYM[a][b]], d, h[d]) for d in R3] for b in R3] for a in R3]
        self.chr = chr_ = [[[0.5 * sum(gu[i][l] * (dg[l][b][a] + dg[l][a][b] - dg[a][b][l]) for l in R3) for b in R3]
                            for a in R3] for i in R3]
        dGh = [[_d1(u[GHX + k], d, h[d]) for d in R3] for k in R3]
        low = [[[sum(g[k][n] * chr_[n][a][b] for n in R3) for b in R3] for a in R3] for k in R3]
        con = [sum(gu[l][m] * chr_[k][l][m] for l in R3 for m in R3) for k in R3]
        mix = [[[sum(gu[l][m] * low[k][b][m] for m in R3) for b in R3] for l in R3] for k in R3]
        self.dchi = dchi = [_d1(u[CHI], d, h[d]) for d in R3]
        hess = _hessian(u[CHI], h)
        cov = [[hess[a][b] - sum(chr_[k][a][b] * dchi[k] for k in R3) for b in R3] for a in R3]
        lap = sum(gu[a][b] * cov[a][b] for a in R3 for b in R3)
        grad2 = sum(gu[a][b] * dchi[a] * dchi[b] for a in R3 for b in R3)
        self.R = [[None] * 3 for _ in R3]
        for a in R3:
            for b in range(a, 3):
                H = _hessian(u[GXX + SYM[a][b]], h)
                r = -0.5 * sum(gu[l][m] * H[l][m] for l in R3 for m in R3)
                for k in R3:
                    r = r + 0.5 * (g[k][a] * dGh[k][b] + g[k][b] * dGh[k][a]) + (Gh[k] - con[k]) * low[k][a][b]
                    r = r + sum(chr_[k][l][a] * mix[k][l][b] + chr_[k][l][b] * mix[k][l][a] for l in R3)
                r = r + 0.5 / (chi + 1e-30) * (cov[a][b] + g[a][b] * lap)
                r = r - 0.25 / (chi * chi + 1e-30) * (dchi[a] * dchi[b] - 3 * g[a][b] * grad2)
                self.R[a][b] = self.R[b][a] = r
        self.Rs = chi * sum(gu[a][b] * self.R[a][b] for a in R3 for b in R3)
        self.Au = [[sum(gu[i][k] * A[k][j] for k in R3) for j in R3] for i in R3]
        self.AA = sum(self.Au[i][j] * self.Au[j][i] for i in R3 for j in R3)


def _exact_rhs(u, h, src=None):
    """Right-hand side with dissipation over the interior of u (22, z, y, x)."""
    prm = ga.CCZ4Params(**PARAMS)
    chi = _inner(u[CHI])
    chi = torch.where(torch.isfinite(chi) & (chi >= 1e-4), chi, torch.full_like(chi, 1e-4))
    q = _Curvature(u, h, chi)
    al, K, Th = (_inner(u[v]) for v in (ALPHA, KTR, THETA))
    be = [_inner(u[BX + a]) for a in R3]
    g, gu, A, Gh, chr_, dchi = q.g, q.gu, q.A, q.Gh, q.chr, q.dchi
    if src is None:
        rho = S = 0.0
        Si, Sij = [0.0] * 3, [[0.0] * 3 for _ in R3]
    else:
        shape = u.shape[1:]
        rho, S = (_inner(src[i].reshape(shape)) for i in (0, 3))
        Si = [_inner(src[1].reshape(-1, 3)[:, a].reshape(shape)) for a in R3]
        Sij = [[_inner(src[2].reshape(-1, 6)[:, SYM[a][b]].reshape(shape)) for b in R3] for a in R3]
    w = 0.5 * (1 + torch.tanh((chi - prm.chi_blend_center) / prm.chi_blend_width))

    def adv(v):
        f, out = u[v], 0.0
        for d in R3:
            t = lambda k: _taps(f, _unit(d, k))  # noqa: E731, B023
            up = [s * (-25 * t(0) + 48 * t(s) - 36 * t(2 * s) + 16 * t(3 * s) - 3 * t(4 * s)) / (12 * h[d])
                  for s in (-1, 1)]
            out = out + be[d] * (w * torch.where(be[d] >= 0, up[0], up[1]) + (1 - w) * _d1(f, d, h[d]))
        return out

    dbe = [[_d1(u[BX + a], d, h[d]) for d in R3] for a in R3]
    div = dbe[0][0] + dbe[1][1] + dbe[2][2]
    dal = [_d1(u[ALPHA], d, h[d]) for d in R3]
    hal = _hessian(u[ALPHA], h)
    DDa = [[hal[a][b] - sum(chr_[k][a][b] * dal[k] for k in R3) for b in R3] for a in R3]
    dK = [_d1(u[KTR], d, h[d]) for d in R3]
    out = [None] * NV
    out[CHI] = 2 / 3 * chi * (al * K - div) + adv(CHI)
    out[ALPHA] = -2 * al * K + adv(ALPHA)
    for a in R3:
        out[BX + a] = 0.75 * Gh[a] - prm.eta * be[a] + adv(BX + a)
    lap = chi * sum(gu[a][b] * DDa[a][b] for a in R3 for b in R3)
    lap = lap - 0.5 * sum(gu[a][b] * dchi[a] * dal[b] for a in R3 for b in R3)
    out[KTR] = (-lap + al * (q.AA + K * K / 3) + 4 * math.pi * al * (rho + S)
                + prm.kappa1 * (1 - prm.kappa2) * al * Th + adv(KTR))
    out[THETA] = (0.5 * al * (q.Rs - q.AA + 2 / 3 * K * K - 16 * math.pi * rho)
                  - al * prm.kappa1 * (2 + prm.kappa2) * Th + adv(THETA))
    raw = {}
    for a in R3:
        for b in range(a, 3):
            i = SYM[a][b]
            lie = lambda T: sum(T[a][k] * dbe[k][b] + T[b][k] * dbe[k][a] for k in R3) - 2 / 3 * T[a][b] * div  # noqa: E731, B023
            out[GXX + i] = -2 * al * A[a][b] + lie(g) + adv(GXX + i)
            raw[i] = (chi * (-DDa[a][b] + al * (q.R[a][b] - 8 * math.pi * Sij[a][b]))
                      + al * (K * A[a][b] - 2 * sum(A[a][k] * q.Au[k][b] for k in R3)) + lie(A) + adv(AXX + i))
    tr = sum(gu[a][b] * raw[SYM[a][b]] for a in R3 for b in R3)
    for a in R3:
        for b in range(a, 3):
            out[AXX + SYM[a][b]] = raw[SYM[a][b]] - g[a][b] * tr / 3
    hbe = [_hessian(u[BX + a], h) for a in R3]
    for a in R3:
        out[GHX + a] = (2 * al * sum(chr_[a][b][c] * A[b][c] for b in R3 for c in R3)
                        - 4 / 3 * al * sum(gu[a][b] * dK[b] for b in R3)
                        - 16 * math.pi * al * sum(gu[a][b] * Si[b] for b in R3)
                        + 3 * al / (chi + 1e-30) * sum(q.Au[a][b] * dchi[b] for b in R3)
                        + sum(gu[b][c] * hbe[a][b][c] for b in R3 for c in R3)
                        + sum(gu[a][b] * hbe[c][c][b] for b in R3 for c in R3) / 3
                        - sum(Gh[b] * dbe[a][b] for b in R3) + 2 / 3 * Gh[a] * div - 2 * prm.kappa1 * al * Gh[a]
                        + adv(GHX + a))
    out = torch.stack(out)
    for d in R3:
        t = lambda k: _taps(u, _unit(d, k))  # noqa: E731, B023
        out += prm.ko_sigma / (64 * h[d]) * (t(-3) + t(3) - 6 * (t(-2) + t(2)) + 15 * (t(-1) + t(1)) - 20 * t(0))
    return out


def _centres(box):
    """Cell centres per axis, on the host: the transfers round positions that lie half way
    between two cells, where a division's last bit decides."""
    n, lo, _ = box
    h = _dx(box)
    return [lo[d] + (torch.arange(n[d] + 2 * NG, dtype=torch.float64) - NG + 0.5) * h[d] for d in R3]


def _side(u, d, k):
    return u.select(3 - d, k if k >= 0 else u.shape[3 - d] + k)


def _exact_fill(u, box, mode, faces=0x3F):
    """Ghost zones in passes over x, y, z, each over the full extent of the other axes."""
    x = [c.cuda() for c in _centres(box)]
    inf = torch.tensor(F_INF, dtype=torch.float64, device="cuda").reshape(-1, 1, 1)
    for d in R3:
        n = box[0][d]
        for q in range(NG):
            for side in (0, 1):
                ghost, edge = (NG - 1 - q, NG) if side == 0 else (NG + n + q, NG + n - 1)
                if mode == ga.BC_PERIODIC:
                    edge = NG + (ghost - NG) % n
                elif mode == ga.BC_OUTFLOW and not faces >> (2 * d + side) & 1:
                    continue
                val = _side(u, d, edge)
                if mode == ga.BC_SOMMERFELD:
                    r2 = [x[2][:, None, None] ** 2, x[1][None, :, None] ** 2, x[0][None, None, :] ** 2]
                    at = lambda k: torch.sqrt(sum((x[d][k] ** 2 if a == d else r2[2 - a].reshape(-1)[:, None] if  # noqa: E731, B023
                                                   a == max(c for c in R3 if c != d) else  # noqa: B023
                                                   r2[2 - a].reshape(-1)[None, :]) for a in R3)) + 1e-30  # noqa: B023
                    val = inf + (val - inf) * at(edge) / at(ghost)
                _side(u, d, ghost).copy_(val)


def _exact_step(u, box, dt, bc, pre, src=None):
    """One SSP-RK3 step of u in place."""
    h = _dx(box)
    if pre is not None:
        _exact_fill(u, box, pre)
    stage = u
    for a1, a2, a3 in ((1.0, 0.0, 1.0), (0.75, 0.25, 0.25), (1 / 3, 2 / 3, 2 / 3)):
        new = a1 * _inner(u) + a2 * _inner(stage) + a3 * dt * _exact_rhs(stage, h, src)
        new[CHI] = torch.where(torch.isfinite(new[CHI]), new[CHI], torch.zeros_like(new[CHI])).clamp(1e-4, 1.5)
        new[ALPHA] = torch.where(torch.isfinite(new[ALPHA]), new[ALPHA], torch.zeros_like(new[ALPHA])).clamp(min=1e-6)
        stage = u.clone()
        if a1 < 0.5:
            xx, xy, xz, yy, yz, zz = new[GXX:GXX + 6]
            det = xx * (yy * zz - yz * yz) - xy * (xy * zz - yz * xz) + xz * (xy * yz - yy * xz)
            new[GXX:GXX + 6] *= det ** (-1.0 / 3.0)
            xx, xy, xz, yy, yz, zz = new[GXX:GXX + 6]
            cof = [yy * zz - yz * yz, xz * yz - xy * zz, xy * yz - xz * yy, xx * zz - xz * xz, xz * xy - xx * yz,
                   xx * yy - xy * xy]
            tr = sum((1 if i in (0, 3, 5) else 2) * cof[i] * new[AXX + i] for i in range(6))
            new[AXX:AXX + 6] -= tr / 3 * new[GXX:GXX + 6]
            stage = u
        _inner(stage).copy_(new)
        _exact_fill(stage, box, bc)


def _exact_prolong(uc, boxc, uf, boxf):
    """Trilinear from the coarse block into every cell of the fine one."""
    idx, wgt = [], []
    for d in R3:
        h = _dx(boxc)[d]
        c = (_centres(boxf)[d] - _centres(boxc)[d][NG]) / h + NG
        c0 = torch.clamp(torch.sign(c) * torch.floor(torch.abs(c) + 0.5), 0, boxc[0][d] + 2 * NG - 1)
        f = c - c0
        c1 = torch.clamp(c0 + torch.where(f >= 0, 1.0, -1.0), 0, boxc[0][d] + 2 * NG - 1)
        idx.append((c0.long().cuda(), c1.long().cuda()))
        wgt.append(((1 - f.abs()).cuda(), f.abs().cuda()))
    out = uc
    for d in R3:
        shape = [-1 if a == 3 - d else 1 for a in range(4)]
        out = sum(out.index_select(3 - d, idx[d][k]) * wgt[d][k].reshape(shape) for k in (0, 1))
    uf.copy_(out)


def _exact_restrict(uf, boxf, uc, boxc):
    """2x2x2 averages of the fine block into the coarse interior cells it covers."""
    at = []
    for d in R3:
        first = (_centres(boxc)[d] - _centres(boxf)[d][0]) / _dx(boxf)[d]
        b = (torch.sign(first) * torch.floor(torch.abs(first) + 0.5)).long() - 1
        c = torch.arange(b.numel())
        ok = (c >= NG) & (c < NG + boxc[0][d]) & (b >= NG) & (b + 2 <= 2 * NG + boxf[0][d])
        at.append((c[ok].cuda(), b[ok].cuda()))
    out = uf
    for d in R3:
        out = out.index_select(3 - d, at[d][1]) + out.index_select(3 - d, at[d][1] + 1)
    uc[:, at[2][0][:, None, None], at[1][0][None, :, None], at[0][0][None, None, :]] = out / 8


def _open_faces(box, parents):
    """Bits of the faces no parent block covers (low side 2d, high side 2d + 1)."""
    mask = 0
    n, _, _ = box
    h = _dx(box)
    for d in R3:
        x = _centres(box)[d]
        ends = [(float(_centres(p)[d][NG]), float(_centres(p)[d][NG + p[0][d] - 1])) for p in parents]
        if not any(a <= float(x[NG]) + 0.5 * h[d] for a, _ in ends):
            mask |= 1 << (2 * d)
        if not any(b >= float(x[NG + n[d] - 1]) - 0.5 * h[d] for _, b in ends):
            mask |= 2 << (2 * d)
    return mask


def _exact_hierarchy(states, geo, dt0):
    def fill(l):
        for u, box in zip(states[l], geo[l]):
            if l == 0:
                _exact_fill(u, box, ga.BC_OUTFLOW)
                continue
            for uc, boxc in zip(states[l - 1], geo[l - 1]):
                _exact_prolong(uc, boxc, u, box)
            faces = _open_faces(box, geo[l - 1])
            if faces:
                _exact_fill(u, box, ga.BC_OUTFLOW, faces)

    # On a finer level the fill after a step (and the one that begins the parent's second
    # substep) sets every cell anew from the parent, so only the last substep's fill is left.
    def cycle(l):
        fill(l)
        if l == 0:
            for u, box in zip(states[l], geo[l]):
                _exact_step(u, box, dt0, ga.BC_SOMMERFELD, None)
            fill(l)
        if l + 1 < len(geo):
            cycle(l + 1)
            for uf, boxf in zip(states[l + 1], geo[l + 1]):
                for uc, boxc in zip(states[l], geo[l]):
                    _exact_restrict(uf, boxf, uc, boxc)

    cycle(0)


def _exact_monitor(u, box):
    """Sums of H^2 and |M|^2 over the interior."""
    h = _dx(box)
    chi, K = _inner(u[CHI]), _inner(u[KTR])
    q = _Curvature(u, h, chi)
    ham = q.Rs + 2 / 3 * K * K - q.AA
    dA = [[[_d1(u[AXX + SYM[a][b]], d, h[d]) for d in R3] for b in R3] for a in R3]
    mom = 0.0
    for a in R3:
        m = -2 / 3 * _d1(u[KTR], a, h[a])
        for b in R3:
            for c in R3:
                DA = dA[c][a][b] - sum(q.chr[k][b][c] * q.A[k][a] + q.chr[k][b][a] * q.A[c][k] for k in R3)
                m = m + q.gu[b][c] * (DA - 3 / (2 * chi + 1e-30) * q.A[a][b] * q.dchi[c])
        mom = mom + float((m * m).sum())
    return float((ham * ham).sum()), mom


def exact(case, seed):
    kind = case["kind"]
    s = prepare(case, seed)
    torch.cuda.synchronize()
    if kind in ("rhs_host", "rhs_device"):
        u = s["u"] if kind == "rhs_device" else torch.from_numpy(s["grid"].array).cuda()
        src = s["src"] and [torch.as_tensor(a).cuda() for a in s["src"]]
        out = torch.zeros_like(u)
        _inner(out).copy_(_exact_rhs(u, _dx(_box(case)), src))
        return out
    geo = _geometry(case)
    states = [[u.clone() for u in lv] for lv in s["out"]]
    if kind == "telemetry":
        sums = [_exact_monitor(u, box) for lv, boxes in zip(states, geo) for u, box in zip(lv, boxes)]
        out = dict(ham=sum(a for a, _ in sums), mom=sum(b for _, b in sums),
                   count=sum(math.prod(n) for lv in geo for n, _, _ in lv))
        for l, (lv, boxes) in enumerate(zip(states, geo)):
            dt = s["dt"] / 2 ** l
            out["cfl%d" % l] = max(float(sum(_inner(u[BX + d]).abs() * dt / _dx(b)[d] for d in R3).max())
                                   for u, b in zip(lv, boxes))
            out["nonfinite%d" % l] = sum(int((~torch.isfinite(_inner(u))).sum()) for u in lv)
        return out
    if kind == "hierarchy":
        _exact_hierarchy(states, geo, s["dt"])
        return [u for lv in states for u in lv]
    dts = s.get("dts", [s["dt"]])
    m = _mode(case)
    for lv, boxes, dt in zip(states, geo, dts):
        for u, box in zip(lv, boxes):
            _exact_step(u, box, dt, m["bc_mode"], m["pre_fill"], s.get("src"))
    return [u for lv in states for u in lv] if kind == "levels" else states[0][0]
