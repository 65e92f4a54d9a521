"""The timestep workloads that libnpbmz is timed on.

A forward case is what a program does with a context: it holds a multi-zone
problem with its fields in HBM, advances it by a run's worth of timesteps and
reads the solution back.  An adjoint case asks for the gradients of a weighted
sum of squares of the final solution.  Sizes are the benchmark classes of
``npbapps_amd.zones`` with their own time steps and counts, and grids between
them that split unevenly.

``exact`` computes the same passes in plain torch, in 64 bits and on the CPU:
the schemes are written as whole-array expressions over a zone, and the
gradients are torch's own.
"""
import functools
import math

import numpy as np
import torch

import npbapps_amd as P
from npbapps_amd import native

# bench, grid, zones, size ratio of the uneven split, time step and step count;
# adjoint cases add the checkpoint interval
_KEYS = ("bench", "gx", "gy", "gz", "xz", "yz", "ratio", "dt", "steps", "ckpt", "mode", "npb")


def _case(name, *values):
    return {"name": name, **dict(zip(_KEYS, values))}


def listed():
    return [
        # the smallest class, a whole run: launches and latencies are all of it
        _case("bt-s", "BT", 24, 24, 6, 2, 2, 3.0, 0.01, 60, 0, "graph", False),
        # the headline run: 64 uneven zones
        _case("bt-b", "BT", 304, 208, 17, 8, 8, 4.5, 0.0003, 200, 0, "graph", False),
        # the largest run: four times class B's points in 256 uneven zones
        _case("bt-c", "BT", 480, 320, 28, 16, 16, 4.5, 0.0001, 200, 0, "graph", False),
        # a grid of a user's own: few zones of odd sizes, launched without graphs
        _case("bt-odd", "BT", 131, 97, 23, 3, 2, 2.2, 0.0003, 100, 0, "batched", False),
        # SP's whole runs: equal zones, few lines in flight (A) and many (B)
        _case("sp-a", "SP", 128, 128, 16, 4, 4, 1.0, 0.0015, 400, 0, "graph", False),
        _case("sp-b", "SP", 304, 208, 17, 8, 8, 1.0, 0.001, 400, 0, "graph", False),
        # LU's whole runs: the library's default exchange planes on small
        # zones, and the verified NPB planes on the ordinary and large ones
        _case("lu-w", "LU", 64, 64, 8, 4, 4, 1.0, 0.0015, 300, 0, "graph", False),
        _case("lu-a", "LU", 128, 128, 16, 4, 4, 1.0, 2.0, 250, 0, "graph", True),
        _case("lu-b", "LU", 304, 208, 17, 4, 4, 1.0, 2.0, 250, 0, "graph", True),
        # gradients through a run, u kept every 20 steps: the benchmark's
        # three adjoint workloads
        _case("bt-a-adjoint", "BT", 128, 128, 16, 4, 4, 4.5, 0.0008, 200, 20, "graph", False),
        _case("sp-a-adjoint", "SP", 128, 128, 16, 4, 4, 1.0, 0.0015, 100, 20, "graph", False),
        _case("lu-a-adjoint", "LU", 128, 128, 16, 4, 4, 1.0, 2.0, 100, 20, "graph", True),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """Another run: any benchmark and direction, 1 to 8 zones a side, zones of
    6 to about 80 points a side, uneven splits (not LU, whose zones are
    equal), with and without graphs."""
    while True:
        bench = rng.choice(["BT", "BT", "SP", "LU"])
        adjoint = rng.random() < 0.3
        xz, yz = rng.randint(1, 8), rng.randint(1, 8)
        nx, ny, gz = _log(rng, 7, 80), _log(rng, 7, 60), _log(rng, 6, 34)
        gx, gy, ratio = xz * nx, yz * ny, 1.0
        if bench != "LU":
            gx, gy = gx + rng.randint(0, xz - 1), gy + rng.randint(0, yz - 1)
            if xz > 1 and yz > 1 and rng.random() < 0.7:
                ratio = round(rng.uniform(1.2, 4.5), 2)
        steps = _log(rng, 10, 200)
        ckpt = min(steps, rng.randint(4, 20)) if adjoint else 0
        mode = "batched" if rng.random() < 0.25 else "graph"
        dt = {"BT": 0.0003, "SP": 0.0007, "LU": 1.0}[bench]
        case = dict(zip(_KEYS, (bench, gx, gy, gz, xz, yz, ratio, dt, steps, ckpt, mode,
                                bench == "LU" and rng.random() < 0.7)))
        smallest = min(_widths(gx, xz, ratio if yz > 1 else 1.0) +
                       _widths(gy, yz, ratio if xz > 1 else 1.0))
        pts = gx * gy * gz
        if smallest >= 6 and pts <= 1_000_000 and pts * steps <= (2e7 if adjoint else 8e7):
            return case


# ------------------------------------------------------------------- inputs
def _widths(n, parts, ratio):
    """Zone widths along one axis: equal, or a geometric progression whose
    largest is `ratio` times its smallest."""
    if abs(ratio - 1.0) > 1e-10 and parts > 1:
        r = math.exp(math.log(ratio) / (parts - 1))
        first = n * (r - 1.0) / (r ** parts - 1.0)
        end = [int(first * (r ** i - 1.0) / (r - 1.0) + 0.45) for i in range(parts + 1)]
    else:
        end = [i * n // parts for i in range(parts + 1)]
    return [b - a for a, b in zip(end, end[1:])]


def _shapes(case):
    """(nz, ny, nx) of every zone, x fastest."""
    ratio = case["ratio"] if case["xz"] > 1 and case["yz"] > 1 else 1.0
    wx, wy = _widths(case["gx"], case["xz"], ratio), _widths(case["gy"], case["yz"], ratio)
    return [(case["gz"], ny, nx) for ny in wy for nx in wx]


_CE = torch.tensor([
    [2.0, 0.0, 0.0, 4.0, 5.0, 3.0, 0.5, 0.02, 0.01, 0.03, 0.5, 0.4, 0.3],
    [1.0, 0.0, 0.0, 0.0, 1.0, 2.0, 3.0, 0.01, 0.03, 0.02, 0.4, 0.3, 0.5],
    [2.0, 2.0, 0.0, 0.0, 0.0, 2.0, 3.0, 0.04, 0.03, 0.05, 0.3, 0.5, 0.4],
    [2.0, 2.0, 0.0, 0.0, 0.0, 2.0, 3.0, 0.03, 0.05, 0.04, 0.2, 0.1, 0.3],
    [5.0, 4.0, 3.0, 2.0, 0.1, 0.4, 0.3, 0.05, 0.04, 0.03, 0.1, 0.3, 0.2]], dtype=torch.float64)


def _solution(shape, h):
    """The benchmarks' steady solution on one zone (nz, ny, nx, 5), points h
    apart: a quartic in each coordinate."""
    out = _CE[:, 0].expand(*shape, 5).clone()
    for axis in range(3):  # x, y, z
        n = shape[2 - axis]
        s = (torch.arange(n, dtype=torch.float64) * h[axis])[:, None]
        poly = s * (_CE[:, 1 + axis] + s * (_CE[:, 4 + axis] + s * (_CE[:, 7 + axis] +
                                                                   s * _CE[:, 10 + axis])))
        out += poly.reshape([n if d == 2 - axis else 1 for d in range(3)] + [5])
    return out


@functools.lru_cache(maxsize=16)
def _steady(bench, gx, gy, gz, xz, yz, ratio, dt):
    """The steady solution and the forcing that balances it, zone by zone."""
    case = dict(zip(_KEYS, (bench, gx, gy, gz, xz, yz, ratio, dt)))
    k, shapes = _Scheme(case), _shapes(case)
    known, fields = {}, []
    for s in shapes:
        if s not in known:
            u = _solution(s, k.h)
            known[s] = (u, _pad(_operator(u, k) * (1.0 if bench == "LU" else -1.0)))
        fields.append(known[s])
    return fields


def _inputs(case, seed):
    """Initial u and the forcing of every zone.  u is the steady solution
    disturbed by smooth waves of up to 6 %, except on the k walls, which hold
    it: a state between a run's first guess and its end."""
    rng = np.random.default_rng(seed)
    u0, forcing = [], []
    for u, f in _steady(*(case[k] for k in _KEYS[:8])):
        nz, ny, nx, _ = u.shape
        wave = 0.0
        for axis, n in ((2, nx), (1, ny), (0, nz)):
            t = torch.linspace(0.0, 1.0, n, dtype=torch.float64)[:, None]
            amp, freq, phase = (torch.from_numpy(rng.uniform(a, b, 5))
                                for a, b in ((0.005, 0.02), (1.0, 9.0), (0.0, 6.28)))
            wave = wave + (amp * torch.sin(freq * t + phase)).reshape(
                [n if d == axis else 1 for d in range(3)] + [5])
        zeta = torch.linspace(0.0, 1.0, nz, dtype=torch.float64).reshape(nz, 1, 1, 1)
        u0.append(u * (1.0 + 4.0 * zeta * (1.0 - zeta) * wave))
        forcing.append(f)
    return u0, forcing


def _weights(case, seed):
    n = 5 * case["gx"] * case["gy"] * case["gz"]
    return np.random.Generator(np.random.Philox(seed)).random(n)


def _flat(zones):
    return np.concatenate([z.numpy().ravel() for z in zones])


# ---------------------------------------------------------------- the passes
def prepare(case, seed):
    zones = P.zone_setup(case["xz"], case["yz"], case["gx"], case["gy"], case["gz"],
                         case["ratio"], use_round=case["bench"] == "LU")
    ctx = P.Context(case["bench"], zones, case["dt"], omega=1.2, npb_exchange=case["npb"])
    u0, forcing = _inputs(case, seed)
    ctx.put_all(native.FIELD_U, _flat(u0))
    ctx.put_all(native.FIELD_FORCING, _flat(forcing))
    if case["bench"] == "LU":
        ctx.run_phase(native.PHASE_RHS)  # an iteration starts from rsd = rhs(u)
    return {"case": case, "ctx": ctx, "w": _weights(case, seed) if case["ckpt"] else None}


def run(state):
    case, ctx = state["case"], state["ctx"]
    if case["ckpt"]:
        r = ctx.adjoint(case["steps"], case["ckpt"], state["w"])
        return {k: r[k] for k in ("loss", "grad_u0", "grad_forcing")}
    ctx.step(case["steps"], case["mode"])
    return {"u": ctx.get_all(native.FIELD_U)}


def work(case):
    """A step reads u and the forcing and writes u: 120 bytes a point; its
    operations are the benchmarks' own counts.  A gradient needs every step
    twice (the states between checkpoints are recomputed), then reads each
    step's u and updates dloss/du and dloss/dforcing; its reverse step is
    counted as two forward ones."""
    zones = P.zone_setup(case["xz"], case["yz"], case["gx"], case["gy"], case["gz"],
                         case["ratio"], use_round=case["bench"] == "LU")
    ops = P.mflops_per_step(case["bench"], zones) * 1e6
    if ops <= 0.0:  # the counting polynomial is for zones of 12 points a side and more
        ops = 1000.0 * zones.npoints
    per_step, ends, times = (440.0, 160.0, 4) if case["ckpt"] else (120.0, 40.0, 1)
    return {"bytes": zones.npoints * (per_step * case["steps"] + ends),
            "flops": times * ops * case["steps"]}


def tolerance(case):
    """About four times what separates the FMA kernels from the ones without
    contraction (u: 5e-17, at most 3e-16 at a point) and the line solves and
    sweeps from their other elimination orders (gradients: 1e-15, at most
    2.4e-14): the steps damp rounding errors, so u stays within an ulp."""
    return {"rel": 4e-15, "max": 1e-13} if case["ckpt"] else {"rel": 3e-16, "max": 4e-15}


# ------------------------------------------- the same passes in plain torch
class _Scheme:
    """Grid spacings, stencil factors and dissipation of one problem."""

    def __init__(self, case):
        self.bench, self.dt, self.omega = case["bench"], case["dt"], 1.2
        if self.bench == "LU":
            n = (case["gx"] // case["xz"], case["gy"] // case["yz"], case["gz"])
            self.h = [1.0 / (m - 1) for m in n]
        else:
            self.h = [1.0 / ((case["gx"] - 1) / case["xz"]), 1.0 / ((case["gy"] - 1) / case["yz"]),
                      1.0 / (case["gz"] - 1)]
        self.t1 = [1.0 / (h * h) for h in self.h]
        self.t2 = [1.0 / (2.0 * h) for h in self.h]
        self.dd = [0.75, 0.75, 1.0]
        self.dssp = 0.25


_C1, _C2, _C34, _C1C5 = 1.4, 0.4, 0.1, 1.96
_C1345 = _C34 * _C1C5


def _along(u, axis, lo, hi):
    """Interior points of a zone, shifted along x, y or z to points lo..n+hi-1."""
    sl = [slice(1, -1)] * 3
    n = u.shape[2 - axis]
    sl[2 - axis] = slice(lo, n + hi)
    return u[tuple(sl)]


def _pad(v):
    """Zeros on a zone's boundary around its interior values."""
    return torch.nn.functional.pad(v, (0, 0, 1, 1, 1, 1, 1, 1))


def _operator(u, k):
    """Flux differences, viscous terms and fourth-order dissipation of
    compute_rhs on a zone's interior."""
    rho = u[..., :1]
    w = u[..., 1:4] / rho
    q = 0.5 * (u[..., 1:4] * w).sum(-1, keepdim=True)  # kinetic energy
    p = _C2 * (u[..., 4:] - q)
    total = 0.0
    for d in range(3):
        wd = w[..., d:d + 1]
        push = torch.zeros(5, dtype=u.dtype)
        push[d + 1] = 1.0
        flux = u * wd + p * push + torch.cat((torch.zeros_like(u[..., :4]), p * wd), -1)
        c = _C34 * k.t1[d]
        scale = torch.full((3,), c, dtype=u.dtype)
        scale[d] *= 4.0 / 3.0
        visc = torch.cat((torch.zeros_like(rho), scale * w,
                          c * ((1.0 - _C1C5) * (q / rho) + wd * wd / 6.0 +
                               _C1C5 * (u[..., 4:] / rho))), -1)
        visc = visc + k.dd[d] * k.t1[d] * u
        total = total - k.t2[d] * (_along(flux, d, 2, 0) - _along(flux, d, 0, -2))
        total = total + (_along(visc, d, 2, 0) - 2.0 * _along(visc, d, 1, -1) +
                         _along(visc, d, 0, -2))
        # fourth difference, cut at the ends of the line: a point next to the
        # boundary weighs 5 and drops that boundary value, a point two off it
        # drops the one beyond
        n = u.shape[2 - d]
        i = torch.arange(1, n - 1).reshape([n - 2 if a == 2 - d else 1 for a in range(3)] + [1])
        wide = torch.nn.functional.pad(u.movedim(2 - d, -1), (1, 1)).movedim(-1, 2 - d)
        total = total - k.dssp * (
            (i >= 3) * _along(wide, d, 0, -4) - 4.0 * (i >= 2) * _along(u, d, 0, -2) +
            torch.where((i == 1) | (i == n - 2), 5.0, 6.0) * _along(u, d, 1, -1) -
            4.0 * (i <= n - 3) * _along(u, d, 2, 0) + (i <= n - 4) * _along(wide, d, 4, 0))
    return total


def _jacobians(u, d):
    """Flux and viscous Jacobians of direction d at every point, (..., 5, 5)."""
    rho, e = u[..., 0], u[..., 4] / u[..., 0]
    w = [u[..., m] / rho for m in (1, 2, 3)]
    wd, ke = w[d], sum(x * x for x in w)
    zero, one = torch.zeros_like(rho), torch.ones_like(rho)
    f = [[zero] * 5 for _ in range(5)]
    n = [[zero] * 5 for _ in range(5)]
    f[0][d + 1] = one
    n[4][0] = -_C1345 * e / rho
    for m in range(3):
        kap = _C34 * (4.0 / 3.0 if m == d else 1.0)
        f[m + 1][0] = -w[m] * wd + (0.5 * _C2 * ke if m == d else 0.0)
        f[m + 1][d + 1] = w[m] * one
        if m != d:
            f[m + 1][m + 1] = wd
            f[d + 1][m + 1] = -_C2 * w[m]
            f[4][m + 1] = -_C2 * w[m] * wd
        n[m + 1][0] = -kap * w[m] / rho
        n[m + 1][m + 1] = kap / rho
        n[4][0] = n[4][0] - (kap - _C1345) * w[m] * w[m] / rho
        n[4][m + 1] = (kap - _C1345) * w[m] / rho
    f[d + 1][d + 1] = (2.0 - _C2) * wd
    f[d + 1][4] = _C2 * one
    f[4][0] = (_C2 * ke - _C1 * e) * wd
    f[4][d + 1] = _C1 * e - 0.5 * _C2 * (ke + 2.0 * wd * wd)
    f[4][4] = _C1 * wd
    n[4][4] = _C1345 / rho
    return tuple(torch.stack([torch.stack(r, -1) for r in m], -2) for m in (f, n))


def _lines(v, d):
    """Interior lines along direction d, the line's points first."""
    sl = [slice(1, -1)] * 3
    sl[2 - d] = slice(None)
    return v[tuple(sl)].movedim(2 - d, 0)


def _block_solve(u, rhs, k, d):
    """Block-tridiagonal solve along d on the interior right-hand side."""
    f, n = _jacobians(_lines(u, d), d)
    a1, a2, eye = k.dt * k.t1[d], k.dt * k.t2[d], torch.eye(5, dtype=u.dtype)
    n = n + k.dd[d] * eye
    r = rhs.movedim(2 - d, 0)
    low, mid, upp = -a2 * f - a1 * n, eye + 2.0 * a1 * n, a2 * f - a1 * n
    cs, rs = [], []
    for row in range(1, f.shape[0] - 1):
        b, v = mid[row], r[row - 1]
        if cs:
            b = b - low[row - 1] @ cs[-1]
            v = v - (low[row - 1] @ rs[-1].unsqueeze(-1)).squeeze(-1)
        x = torch.linalg.solve(b, torch.cat((upp[row + 1], v.unsqueeze(-1)), -1))
        cs.append(x[..., :5])
        rs.append(x[..., 5])
    out = [rs[-1]]
    for c, v in zip(cs[-2::-1], rs[-2::-1]):
        out.append(v - (c @ out[-1].unsqueeze(-1)).squeeze(-1))
    return torch.stack(out[::-1]).movedim(0, 2 - d)


def _speed(u):
    return torch.sqrt(_C1 * _C2 / u[..., 0] *
                      (u[..., 4] - 0.5 * (u[..., 1:4] ** 2).sum(-1) / u[..., 0]))


def _penta_solve(u, rhs, k, d):
    """SP's three scalar pentadiagonal systems along d: components 1..3, 4, 5."""
    ul = _lines(u, d)
    rho = _C34 / ul[..., 0]
    dd = k.dd[d]
    # the largest of the direction's four diffusion bounds; each velocity
    # component's width is the direction's own
    width = torch.maximum(torch.maximum(dd + 4.0 / 3.0 * rho, dd + _C1C5 * rho), dd + rho)
    a1, a2 = k.dt * k.t1[d], k.dt * k.t2[d]
    sign = torch.tensor([0.0, 0.0, 0.0, 1.0, -1.0], dtype=u.dtype)
    vel = (ul[..., d + 1] / ul[..., 0]).unsqueeze(-1) + sign * _speed(ul).unsqueeze(-1)
    width = width.unsqueeze(-1)
    r = rhs.movedim(2 - d, 0)
    n, c = ul.shape[0], k.dt * k.dssp
    rows = []
    for i in range(1, n - 1):
        e = [c * (i >= 3), -a2 * vel[i - 1] - a1 * width[i - 1] - 4.0 * c * (i >= 2),
             1.0 + 2.0 * a1 * width[i] + c * (5.0 if i in (1, n - 2) else 6.0),
             a2 * vel[i + 1] - a1 * width[i + 1] - 4.0 * c * (i <= n - 3), c * (i <= n - 4)]
        v = r[i - 1]
        if len(rows) > 1:  # row i-2
            p = rows[-2]
            e[1], e[2], v = e[1] - e[0] * p[0], e[2] - e[0] * p[1], v - e[0] * p[2]
        if rows:
            p = rows[-1]
            e[2], e[3], v = e[2] - e[1] * p[0], e[3] - e[1] * p[1], v - e[1] * p[2]
        rows.append((e[3] / e[2], e[4] / e[2], v / e[2]))
    out = []
    for i in range(len(rows) - 1, -1, -1):
        x = rows[i][2]
        if len(out) > 0:
            x = x - rows[i][0] * out[-1]
        if len(out) > 1:
            x = x - rows[i][1] * out[-2]
        out.append(x)
    return torch.stack(out[::-1]).movedim(0, 2 - d)


def _sp_sweep(u, r, k):
    """txinvr, the three solves and their inverse transforms."""
    ui = u[1:-1, 1:-1, 1:-1]
    rho, bt = ui[..., 0], math.sqrt(0.5)
    w1, w2, w3 = (ui[..., m] / rho for m in (1, 2, 3))
    ke, ac = 0.5 * (w1 * w1 + w2 * w2 + w3 * w3), _speed(ui)
    r1, r2, r3, r4, r5 = r.unbind(-1)
    t1 = _C2 / (ac * ac) * (ke * r1 - w1 * r2 - w2 * r3 - w3 * r4 + r5)
    t2 = bt / rho * (w1 * r1 - r2)
    t3 = bt / rho * ac * t1
    r = torch.stack((r1 - t1, -(w3 * r1 - r4) / rho, (w2 * r1 - r3) / rho, -t2 + t3, t2 + t3), -1)
    r1, r2, r3, r4, r5 = _penta_solve(u, r, k, 0).unbind(-1)
    t1, t2 = bt * r3, 0.5 * (r4 + r5)
    r = torch.stack((-r2, r1, bt * (r4 - r5), -t1 + t2, t1 + t2), -1)
    r1, r2, r3, r4, r5 = _penta_solve(u, r, k, 1).unbind(-1)
    t1, t2 = bt * r1, 0.5 * (r4 + r5)
    r = torch.stack((bt * (r4 - r5), -r3, r2, -t1 + t2, t1 + t2), -1)
    r1, r2, r3, r4, r5 = _penta_solve(u, r, k, 2).unbind(-1)
    t1 = bt * rho / ac * (r4 + r5)
    t2, t3 = r3 + t1, bt * rho * (r4 - r5)
    return torch.stack((t2, -rho * r2 + w1 * t2, rho * r1 + w2 * t2, w3 * t2 + t3,
                        rho * (-w1 * r2 + w2 * r1) + ke * t2 + 2.5 * ac * ac * t1 + w3 * t3), -1)


def _exchange(us, case):
    """Every zone's x and y faces from its neighbours' planes next to them."""
    xz, yz, bench = case["xz"], case["yz"], case["bench"]
    if bench != "LU" and xz * yz == 1:
        return us
    ks = slice(0, -2) if bench == "LU" and not case["npb"] else slice(1, -1)
    got = []
    for z, u in enumerate(us):
        i, j = z % xz, z // xz
        west, east = us[(i - 1) % xz + j * xz], us[(i + 1) % xz + j * xz]
        south, north = us[i + (j - 1) % yz * xz], us[i + (j + 1) % yz * xz]
        if bench == "SP":
            south, north = north, south
        v = u[ks]
        across = slice(None) if bench == "LU" else slice(1, -1)

        def face(own, other):  # LU's j faces own the zone's corners
            return other if bench == "LU" else torch.cat((own[:, :1], other[:, across],
                                                          own[:, -1:]), 1)
        low = face(v[:, 0], south[ks][:, -2]).unsqueeze(1)
        high = face(v[:, -1], north[ks][:, 1]).unsqueeze(1)
        body = torch.cat((west[ks][:, 1:-1, -2:-1], v[:, 1:-1, 1:-1], east[ks][:, 1:-1, 1:2]), 2)
        v = torch.cat((low, body, high), 1)
        got.append(torch.cat((u[:ks.start], v, u[ks.stop:]), 0))
    return got


@functools.lru_cache(maxsize=4)
def _hyperplanes(shape):
    """Indexes of the interior points of each plane i + j + k = const."""
    nz, ny, nx = shape
    k, j, i = np.meshgrid(range(1, nz - 1), range(1, ny - 1), range(1, nx - 1), indexing="ij")
    s = (i + j + k).ravel()
    at = ((k * ny + j) * nx + i).ravel()
    return [torch.from_numpy(at[s == q]) for q in range(3, int(s.max()) + 1)]


def _ssor(us, rsd, k):
    """One lower and one upper sweep over zones of one shape, stacked:
    new u."""
    u, r = torch.stack(us), torch.stack(rsd)
    nzn, (nz, ny, nx) = len(us), u.shape[1:4]
    stride, eye = (1, nx, nx * ny), torch.eye(5, dtype=u.dtype)
    diag, low, upp = eye, [], []
    for d in range(3):
        f, n = _jacobians(u, d)
        n = k.dt * k.t1[d] * (n + k.dd[d] * eye)
        f = k.dt * k.t2[d] * f
        diag = diag + 2.0 * n
        low.append((-f - n).reshape(nzn, -1, 5, 5))
        upp.append((f - n).reshape(nzn, -1, 5, 5))
    inv = torch.linalg.inv(diag).reshape(nzn, -1, 5, 5)
    r = r.reshape(nzn, -1, 5)
    planes = _hyperplanes((nz, ny, nx))

    def sweep(src, blocks, step, order, lower):
        # each plane's new values gathered from the planes before it
        new = src
        for at in order:
            acc = 0.0
            for d in (2, 1, 0):
                nb = at + step * stride[d]
                acc = acc + (blocks[d][:, nb] @ new[:, nb].unsqueeze(-1))
            if lower:
                v = inv[:, at] @ (k.dt * src[:, at].unsqueeze(-1) - k.omega * acc)
            else:
                v = src[:, at].unsqueeze(-1) - inv[:, at] @ (k.omega * acc)
            new = new.index_copy(1, at, v.squeeze(-1))
        return new

    r = sweep(r, low, -1, planes, True)
    r = sweep(r, upp, 1, planes[::-1], False)
    r = r.reshape(u.shape)[:, 1:-1, 1:-1, 1:-1] / (k.omega * (2.0 - k.omega))
    return [a + _pad(b) for a, b in zip(us, r)]


def _advance(us, forcing, case):
    """The case's timesteps from us."""
    k = _Scheme(case)
    if k.bench == "LU":
        rsd = [_pad(_operator(u, k)) - f for u, f in zip(us, forcing)]
        for _ in range(case["steps"]):
            us = _exchange(us, case)
            us = _ssor(us, rsd, k)
            rsd = [_pad(_operator(u, k)) - f for u, f in zip(us, forcing)]
        return us
    for _ in range(case["steps"]):
        us = _exchange(us, case)
        new = []
        for u, f in zip(us, forcing):
            r = k.dt * (_operator(u, k) + f[1:-1, 1:-1, 1:-1])
            if k.bench == "SP":
                r = _sp_sweep(u, r, k)
            else:
                for d in range(3):
                    r = _block_solve(u, r, k, d)
            new.append(u + _pad(r))
        us = new
    return us


def exact(case, seed):
    """run()'s outputs in plain torch; None where that is long (each step of a
    zone is some hundreds of whole-array operations per row or hyperplane)."""
    points, zones = case["gx"] * case["gy"] * case["gz"], case["xz"] * case["yz"]
    if case["bench"] == "LU":
        rows = 2 * (case["gx"] // case["xz"] + case["gy"] // case["yz"] + case["gz"])
    else:
        rows = case["gx"] * case["yz"] + case["gy"] * case["xz"] + case["gz"] * zones
    cost = case["steps"] * (rows * 5e-4 + points * 1e-5) * (4 if case["ckpt"] else 1)
    if cost > 15.0:
        return None
    u0, forcing = _inputs(case, seed)
    if not case["ckpt"]:
        return {"u": _flat(_advance(u0, forcing, case))}
    for t in u0:
        t.requires_grad_()
    forcing = [f.clone().requires_grad_() for f in forcing]
    us = _advance(u0, forcing, case)
    w = torch.from_numpy(_weights(case, seed))
    loss = (w * torch.cat([u.reshape(-1) for u in us]) ** 2).sum()
    g = torch.autograd.grad(loss, u0 + forcing)
    return {"loss": float(loss.detach()), "grad_u0": _flat(g[:len(u0)]),
            "grad_forcing": _flat(g[len(u0):])}
