"""The workloads by which this framework's speed is followed, over the range of its use.

Each case goes through the public operator surface: `Mult` (one right-hand
side, what another ODE solver calls), `Step` (one SSP-RK3 step), `Run` (the
time loop on the device) and `Ensemble.Step`.  listed() gives the followed
cases, draw() one more of the same ranges, prepare() the operator and states a
program has in hand, run() one pass, work() its algorithmic bytes and flops,
and exact() the same result from a plain torch FP64 evaluation of the scheme
(structured element grids, general per-node metrics) that shares no code with
the library.

A case's keys: grid ("box", "quad", "hex" or "ensemble"), order, the elements
per direction nx, ny, nz (0: direction absent), flow (the kind of state),
ns (Navier-Stokes), blend (indicator and subcell blending), mixed, entry
("mult", "step" or "run") and steps (time steps per pass).
"""
import math

import numpy as np
import torch

from prandtl_amd import DGSEMOperator
from prandtl_amd.operator import Ensemble, HexMesh, QuadMesh

GAMMA = 1.4
PR = 0.71
MU = 1.0 / 1600.0


def _c(name, grid, order, nx, ny, nz, flow, entry, ns=False, blend=False, mixed=False, steps=1):
    c = dict(name=name, grid=grid, order=order, nx=nx, ny=ny, nz=nz, flow=flow, entry=entry, ns=ns, blend=blend,
             mixed=mixed, steps=steps)
    if not name:
        del c["name"]
    return c


def listed():
    return [
        # a 1-D shock tube (Sod's elements) in the device time loop: every
        # launch is one workgroup's chain of phases
        _c("tube1d_run", "box", 3, 128, 0, 0, "tube", "run", blend=True, steps=32),
        # one right-hand side of the isentropic-vortex mesh: the smallest call
        _c("vortex2d_mult", "box", 3, 16, 16, 0, "smooth", "mult"),
        # the Kelvin-Helmholtz shear layer, shock capturing on, stepped with
        # a fixed step
        _c("shear2d_step", "box", 4, 64, 64, 0, "shear", "step", blend=True, steps=4),
        # the triple-point problem's box with slip walls in the time loop
        _c("triple2d_run", "box", 3, 112, 48, 0, "blast", "run", blend=True, steps=16),
        # a supersonic channel on a distorted quadrilateral mesh (as many
        # elements as the forward-facing step refined once), inflow, outflow
        # and slip walls
        _c("channel2d_quad_mult", "quad", 3, 170, 80, 0, "channel", "mult", blend=True),
        # a large 2-D blended run (the double Mach reflection's element count)
        _c("shear2d_large_mult", "box", 3, 384, 384, 0, "shear", "mult", blend=True),
        # the Taylor-Green vortex at the headline's size
        _c("tgv3d_n3_step", "box", 3, 16, 16, 16, "tgv", "step", ns=True, steps=4),
        # the same in the mixed-precision form
        _c("tgv3d_n3_mixed_step", "box", 3, 16, 16, 16, "tgv", "step", ns=True, mixed=True, steps=4),
        # a larger box of odd sizes: throughput instead of latency
        _c("tgv3d_n3_large_mult", "box", 3, 45, 43, 41, "tgv", "mult", ns=True),
        # the large high-order run with blending: the largest case
        _c("tgv3d_n7_mult", "box", 7, 32, 32, 32, "tgv", "mult", ns=True, blend=True),
        # the Taylor-Green vortex on warped hexahedra
        _c("tgv3d_hex_mult", "hex", 3, 16, 16, 16, "tgv", "mult", ns=True),
        # 64 independent 2-D cases of orders 2..5, half of them blended
        _c("ensemble64_step", "ensemble", 0, 64, 0, 0, "mixed", "step", steps=2),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["tube", "box2", "box2", "box2open", "quad", "box3", "box3", "box3", "box3high", "hex",
                       "ensemble"])
    if kind == "tube":
        return _c("", "box", rng.randint(1, 7), _log(rng, 32, 4096), 0, 0, "tube", "run", blend=True,
                  steps=rng.randint(8, 40))
    if kind == "ensemble":
        return _c("", "ensemble", 0, rng.randint(4, 64), 0, 0, "mixed", "step", steps=rng.randint(1, 2))
    if kind in ("box2", "box2open", "quad"):
        nx, ny = _log(rng, 12, 400), _log(rng, 12, 400)
        if kind == "quad":
            return _c("", "quad", rng.randint(1, 5), min(nx, 200), min(ny, 200), 0, "channel", "mult",
                      blend=rng.random() < 0.8)
        if kind == "box2open":
            return _c("", "box", rng.randint(2, 4), nx, ny, 0, "blast", "run", blend=True, steps=rng.randint(4, 20))
        blend = rng.random() < 0.6
        return _c("", "box", rng.randint(2, 5), nx, ny, 0, "shear" if blend else "smooth",
                  rng.choice(["mult", "step"]), blend=blend, steps=rng.randint(1, 4))
    if kind == "hex":
        return _c("", "hex", rng.randint(2, 4), _log(rng, 4, 24), _log(rng, 4, 24), _log(rng, 4, 24), "tgv", "mult",
                  ns=rng.random() < 0.7, blend=rng.random() < 0.3)
    if kind == "box3high":
        return _c("", "box", rng.randint(5, 7), _log(rng, 4, 22), _log(rng, 4, 22), _log(rng, 4, 22), "tgv", "mult",
                  ns=rng.random() < 0.6, blend=rng.random() < 0.6)
    ns = rng.random() < 0.7
    mixed = ns and rng.random() < 0.2
    return _c("", "box", rng.randint(2, 4), _log(rng, 5, 48), _log(rng, 5, 48), _log(rng, 5, 48), "tgv",
              "step" if mixed else rng.choice(["mult", "step"]), ns=ns, blend=rng.random() < 0.3, mixed=mixed,
              steps=rng.randint(1, 4))


# ---------------------------------------------------------------------------
# grids and states
# ---------------------------------------------------------------------------

def _lgl(N):
    """LGL nodes and weights on [0, 1] (roots of (1 - x^2) P_N'(x))."""
    P = np.polynomial.legendre.Legendre.basis(N)
    x = np.concatenate([[-1.0], np.sort(P.deriv().roots().real), [1.0]])
    for _ in range(3):   # Newton on (1 - x^2) P_N'
        dP, d2P = P.deriv()(x[1:-1]), P.deriv(2)(x[1:-1])
        x[1:-1] -= dP / d2P
    w = 2.0 / (N * (N + 1) * P(x) ** 2)
    return 0.5 * (x + 1.0), 0.5 * w


def _dim(c):
    return 1 if c["ny"] == 0 else 2 if c["nz"] == 0 else 3


def _dev():
    return torch.device("cuda:0" if torch.cuda.is_available() else "cpu")


_BOX = {"tube": ((0.0,), (1.0,)), "shear": ((-1.0, -1.0), (1.0, 1.0)), "blast": ((0.0, 0.0), (7.0, 3.0)),
        "smooth": ((-5.0, -5.0), (5.0, 5.0)), "channel": ((0.0, 0.0), (3.0, 1.0)),
        "tgv": ((0.0,) * 3, (2 * math.pi,) * 3)}


def _n(c):
    return (c["nx"], c["ny"], c["nz"])[:_dim(c)]


def _vertices(c, seed):
    """Vertex coordinates of a distorted grid: [dim][(nz+1)][ny+1][nx+1].
    quad: interior vertices moved at random by up to a tenth of an element;
    hex: a smooth periodic warp of a tenth of an element."""
    lo, hi = _BOX[c["flow"]]
    n = _n(c)
    d = len(n)
    rng = np.random.default_rng(seed + 17)
    ax = [np.linspace(lo[r], hi[r], n[r] + 1) for r in range(d)]
    X = np.stack(np.meshgrid(*ax[::-1], indexing="ij")[::-1])
    h = [(hi[r] - lo[r]) / n[r] for r in range(d)]
    if c["grid"] == "quad":
        for r in range(d):
            X[r, 1:-1, 1:-1] += 0.1 * h[r] * rng.uniform(-1, 1, X[r, 1:-1, 1:-1].shape)
        return X
    Y = X.copy()
    for r in range(d):
        e = (r + 1) % d
        Y[r] += 0.1 * h[r] * np.sin(2 * np.pi * (X[e] - lo[e]) / (hi[e] - lo[e]) + rng.uniform(0, 2 * np.pi))
    return Y


def _corners(X):
    """[dim] dicts corner-bit tuple (i, j[, k]) -> element array of a vertex grid."""
    d = X.shape[0]
    out = {}
    for m in range(2 ** d):
        bits = tuple((m >> r) & 1 for r in range(d))
        sl = tuple(slice(1, None) if bits[r] else slice(None, -1) for r in reversed(range(d)))
        out[bits] = np.stack([X[a][sl] for a in range(d)], axis=-1)   # [nz][ny][nx][dim]
    return out


def _coords(c, seed):
    """Node coordinates, a list of dim tensors shaped [nz][ny][nx][Np][Np][Np]
    (x fastest in both groups), and the grid's vertices (None on a box)."""
    dev = _dev()
    n, d, Np = _n(c), _dim(c), c["order"] + 1
    x = torch.tensor(_lgl(c["order"])[0], device=dev)
    shape = tuple(reversed(n)) + (Np,) * d

    def along(v, axis):
        s = [1] * (2 * d)
        s[axis] = v.numel()
        return v.reshape(s)
    lo, hi = _BOX[c["flow"]]
    if c["grid"] == "box":
        X = []
        for r in range(d):
            e = torch.arange(n[r], device=dev, dtype=torch.float64)
            h = (hi[r] - lo[r]) / n[r]
            X.append((lo[r] + h * (along(e, d - 1 - r) + along(x, 2 * d - 1 - r))).expand(shape))
        return X, None
    V = _vertices(c, seed)
    X = [torch.zeros(shape, device=dev, dtype=torch.float64) for _ in range(d)]
    for bits, p in _corners(V).items():
        N = 1.0
        for r in range(d):
            N = N * along(x if bits[r] else 1.0 - x, 2 * d - 1 - r)
        P = torch.tensor(p, device=dev)
        for a in range(d):
            X[a] += N * P[..., a].reshape(tuple(reversed(n)) + (1,) * d)
    return X, V


CHANNEL_IN = (1.4, 2.0, 0.0, 1.0)   # rho, u, v, p: Mach 2


def _tube(seed):
    """Left and right (rho, u, p) and the jump's place of a shock tube."""
    rng = np.random.default_rng(seed + 5)
    L = (1.0 * rng.uniform(0.8, 1.2), rng.uniform(0.0, 0.7), 1.0 * rng.uniform(0.8, 1.2))
    R = (0.125 * rng.uniform(0.8, 1.5), 0.0, 0.1 * rng.uniform(0.8, 1.2))
    return L, R, rng.uniform(0.4, 0.6)


def _cons(rho, vel, p):
    ke = sum(v * v for v in vel)
    return torch.stack([rho] + [rho * v for v in vel] + [p / (GAMMA - 1.0) + 0.5 * rho * ke])


def _state(c, seed):
    """The conservative state [nv][elements][nodes] of a case's flow."""
    X, _ = _coords(c, seed)
    d, flow = _dim(c), c["flow"]
    rng = np.random.default_rng(seed + 101)
    lo, hi = _BOX[flow]
    th = [2 * math.pi * (X[r] - lo[r]) / (hi[r] - lo[r]) for r in range(d)]

    def field(amp):
        f = torch.zeros_like(X[0])
        for _ in range(3):
            k = rng.integers(1, 3, size=d)
            f = f + float(rng.uniform(-1, 1)) * torch.sin(float(rng.uniform(0, 2 * np.pi)) +
                                                          sum(float(k[r]) * th[r] for r in range(d)))
        return (amp / 3.0) * f
    one = torch.ones_like(X[0])
    if flow == "tube":
        L, R, x0 = _tube(seed)
        left = X[0] < x0
        q = [torch.where(left, one * a, one * b) for a, b in zip(L, R)]
        return _cons(q[0], [q[1]], q[2])
    if flow == "smooth":
        return _cons(one + field(0.3), [one + field(1.0) for _ in range(d)], one + field(0.3))
    if flow == "shear":
        s = float(rng.uniform(10, 20))
        B = torch.tanh(s * X[1] + 0.5 * s) - torch.tanh(s * X[1] - 0.5 * s)
        g = torch.Generator(device=X[0].device)
        g.manual_seed(seed + 7)
        noise = torch.rand(X[0].shape, generator=g, device=X[0].device, dtype=torch.float64)
        v = 0.1 * torch.sin(2 * math.pi * X[0] + float(rng.uniform(0, 2 * np.pi))) + 1e-3 * (2.0 * noise - 1.0)
        return _cons(0.5 + 0.75 * B, [0.5 * (B - 1.0), v], one)
    if flow == "blast":
        x0, y0 = float(rng.uniform(0.8, 1.2)), float(rng.uniform(1.3, 1.7))
        left, low = X[0] <= x0, X[1] <= y0
        rho = torch.where(left, one, torch.where(low, one, 0.125 * one))
        p = torch.where(left, one, 0.1 * one)
        return _cons(rho, [0.0 * one, 0.0 * one], p)
    if flow == "channel":
        # a Mach 2 stream with waves and one steep oblique compression
        x0 = float(rng.uniform(0.8, 1.6))
        jump = 0.5 * (1.0 + torch.tanh((X[0] - x0 - 0.5 * X[1]) / 0.01))
        r0, u0, _, p0 = CHANNEL_IN
        return _cons(r0 * (1.0 + 0.8 * jump + field(0.05)), [u0 * (1.0 - 0.25 * jump) + field(0.05), 0.3 * jump + field(0.05)],
                     p0 * (1.0 + 1.4 * jump + field(0.05)))
    # Taylor-Green vortex at Mach 0.1 with density and pressure waves; blended
    # cases also carry a steep density front across part of the box
    x, y, z = X
    u = torch.sin(x) * torch.cos(y) * torch.cos(z) + field(0.05)
    v = -torch.cos(x) * torch.sin(y) * torch.cos(z) + field(0.05)
    w = field(0.1)
    p0 = 1.0 / (GAMMA * 0.01)
    p = p0 + (torch.cos(2 * x) + torch.cos(2 * y)) * (torch.cos(2 * z) + 2.0) / 16.0 + field(0.2)
    rho = one + field(0.02)
    if c["blend"]:
        a = float(rng.uniform(0, 2 * np.pi))
        rho = rho + 0.1 * torch.tanh(torch.sin(x + a) / 0.02) * (1.0 + torch.cos(z)) * 0.5
    return _cons(rho, [u, v, w], p)


def _alpha_max(c):
    return 0.1 if _dim(c) == 3 else 0.5


def _hmin(c):
    lo, hi = _BOX[c["flow"]]
    return min((hi[r] - lo[r]) / m for r, m in enumerate(_n(c)))


_SPEED = {"tube": 2.5, "smooth": 4.0, "shear": 4.0, "blast": 2.0, "channel": 5.0, "tgv": 12.0}


def _dt(c):
    """A fixed step: CFL 0.25 of a bound of the flow's wave speed."""
    return 0.25 * _hmin(c) / (_SPEED[c["flow"]] * (c["order"] + 1) ** 2)


def _box_bc(c, seed):
    if c["flow"] == "tube":
        L, R, _ = _tube(seed)
        ends = []
        for q in (L, R):
            ends.append((q[0], q[0] * q[1], q[2] / (GAMMA - 1.0) + 0.5 * q[0] * q[1] * q[1]))
        return [("specified-state", "specified-state")], [tuple(ends)]
    if c["flow"] == "blast":
        return [("slip", "slip"), ("slip", "slip")], None
    return None, None


def _members(c, seed):
    """The cases of an ensemble: square meshes of 8..64 elements a side,
    orders 2..5, the second half blended shear layers."""
    rng = np.random.default_rng(20261202)   # the ensemble's make-up is the case's; its states are the seed's
    out = []
    for i in range(c["nx"]):
        n = int(rng.choice([8, 16, 24, 32, 48, 64]))
        N = int(rng.integers(2, 6))
        shear = i >= c["nx"] // 2
        out.append(_c("", "box", N, n, n, 0, "shear" if shear else "smooth", "step", blend=shear, steps=c["steps"]))
    return [(m, seed * 1000 + i) for i, m in enumerate(out)]


# ---------------------------------------------------------------------------
# the program
# ---------------------------------------------------------------------------

def _params(c):
    p = dict(gamma=GAMMA, blending=bool(c["blend"]), alpha_max=_alpha_max(c), alpha_min=0.001, quirks=False)
    if c["ns"]:
        p.update(parabolic=True, mu=MU, Pr=PR)
    if c["mixed"]:
        p.update(precision="mixed")
    return p


def _channel_cons():
    r0, u0, v0, p0 = CHANNEL_IN
    return (r0, r0 * u0, r0 * v0, p0 / (GAMMA - 1.0) + 0.5 * r0 * (u0 * u0 + v0 * v0))


def _operator(c, seed):
    lo, hi = _BOX[c["flow"]]
    if c["grid"] == "box":
        bc, st = _box_bc(c, seed)
        return DGSEMOperator(dim=_dim(c), order=c["order"], nelem=_n(c), lo=lo, hi=hi, bc=bc, bc_state=st, **_params(c))
    V = _vertices(c, seed)
    if c["grid"] == "quad":
        nx, ny = _n(c)
        vid = np.arange((nx + 1) * (ny + 1)).reshape(ny + 1, nx + 1)
        elem = np.stack([vid[:-1, :-1], vid[:-1, 1:], vid[1:, 1:], vid[1:, :-1]], axis=-1).reshape(-1, 4)
        sides = [np.stack([vid[:-1, 0], vid[1:, 0]], -1), np.stack([vid[:-1, -1], vid[1:, -1]], -1),
                 np.stack([vid[0, :-1], vid[0, 1:]], -1), np.stack([vid[-1, :-1], vid[-1, 1:]], -1)]
        mesh = QuadMesh(V.reshape(2, -1).T, elem, np.concatenate(sides),
                        np.concatenate([np.full(len(s), i + 1) for i, s in enumerate(sides)]))
        bc = {1: ("supersonic-inflow", _channel_cons()), 2: "supersonic-outflow", 3: "slip", 4: "slip"}
        return DGSEMOperator.quad(mesh, c["order"], bc=bc, **_params(c))
    nx, ny, nz = _n(c)
    vid = np.arange(nx * ny * nz).reshape(nz, ny, nx)
    order = ((0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1))
    elem = np.stack([np.roll(vid, (-k, -j, -i), (0, 1, 2)) for i, j, k in order], axis=-1).reshape(-1, 8)
    cs = _corners(V)
    ec = np.stack([cs[b] for b in order], axis=-2).reshape(-1, 8, 3)
    return DGSEMOperator.hex(HexMesh(np.zeros((nx * ny * nz, 3)), elem, None, None, ec), c["order"], **_params(c))


def prepare(case, seed):
    c = case
    s = dict(c=c, stream=torch.cuda.Stream() if c["entry"] != "mult" else None)
    if c["grid"] == "ensemble":
        ms = _members(c, seed)
        us = [_state(m, sd).reshape(-1) for m, sd in ms]
        s["u0"] = torch.cat(us)
        s["u"] = torch.empty_like(s["u0"])
        s["us"] = list(s["u"].split([u.numel() for u in us]))
        s["dts"] = [_dt(m) for m, _ in ms]
        cases = []
        for m, _ in ms:
            lo, hi = _BOX[m["flow"]]
            cases.append(dict(dim=2, order=m["order"], nelem=_n(m), lo=lo, hi=hi, **_params(m)))
        s["op"] = Ensemble(cases)
        return s
    s["op"] = _operator(c, seed)
    s["u0"] = _state(c, seed).reshape(-1).contiguous()
    s["u"] = torch.empty_like(s["u0"])
    s["dt"] = _dt(c)
    return s


def run(state):
    s = state
    c, op, u = s["c"], s["op"], s["u"]
    if c["entry"] == "mult":
        op.Mult(s["u0"], u)
        return u
    with torch.cuda.stream(s["stream"]):
        u.copy_(s["u0"])
        if c["grid"] == "ensemble":
            for _ in range(c["steps"]):
                op.Step(s["us"], s["dts"])
            return s["us"]
        if c["entry"] == "step":
            for _ in range(c["steps"]):
                op.Step(u, s["dt"])
            return u
        # a run from the initial state: the running wave speed starts anew
        op.GetMaxCharSpeed(reset=True)
        t, n = op.Run(u, 0.0, 1e9, cfl=0.5, max_steps=c["steps"])
        return {"u": u, "t": t, "n": n}


def _flops(c):
    """Flops per node of one right-hand side of the scheme: two-point fluxes
    of the symmetric pairs, surface points (once per face point), the
    indicator, and with Navier-Stokes the lifting and viscous terms."""
    d, Np = _dim(c), c["order"] + 1
    nv = d + 2
    f = d * (Np - 1) / 2 * (45 + 6 * d + 4 * nv) + d / Np * (75 + 12 * d + 4 * nv) + 20
    if c["blend"]:
        f += d * 2 * Np + 15
    if c["ns"]:
        f += 2 * d * Np * (2 * nv - 1) + d / Np * 10 * nv + 30 + 40 * d
    return f


def work(case):
    c = case
    if c["grid"] == "ensemble":
        ws = [work(m) for m, _ in _members(c, 0)]
        return {"bytes": sum(w["bytes"] for w in ws), "flops": sum(w["flops"] for w in ws)}
    d = _dim(c)
    nodes = math.prod(_n(c)) * (c["order"] + 1) ** d
    nv = d + 2
    if c["entry"] == "mult":
        return {"bytes": 16.0 * nv * nodes, "flops": _flops(c) * nodes}
    # a step is three right-hand sides, each of the whole state: read it,
    # write the stage, and read the step's first state in two of them
    rhs = 3 * c["steps"] + (1 if c["entry"] == "run" else 0)
    return {"bytes": 8.0 * nv * nodes * (8 * c["steps"] + (2 if c["entry"] == "run" else 0)),
            "flops": _flops(c) * nodes * rhs}


# ---------------------------------------------------------------------------
# the scheme in plain torch FP64
# ---------------------------------------------------------------------------

class _Scheme:
    """The DGSEM right-hand side on a structured grid of elements with
    general per-node metrics Ja[r][a] (floats on a box)."""

    def __init__(self, c, seed):
        self.c, self.d, self.Np = c, _dim(c), c["order"] + 1
        d, Np = self.d, self.Np
        self.dev = _dev()
        x, w = _lgl(c["order"])
        wb = np.array([1.0 / np.prod([x[i] - x[j] for j in range(Np) if j != i]) for i in range(Np)])
        D = np.zeros((Np, Np))
        for i in range(Np):
            for j in range(Np):
                if i != j:
                    D[i, j] = wb[j] / wb[i] / (x[i] - x[j])
            D[i, i] = -D[i].sum()
        Dh = D.copy()
        Dh[0, 0] += 1.0 / w[0]
        Dh[-1, -1] -= 1.0 / w[-1]
        self.w = w
        T = lambda m: torch.tensor(m, device=self.dev, dtype=torch.float64)  # noqa: E731
        self.D, self.Dh = T(D), T(Dh)
        A, B = np.triu_indices(Np, 1)
        M = np.zeros((Np, len(A)))   # node sums of the symmetric pairs
        for p, (a, b) in enumerate(zip(A, B)):
            M[a, p], M[b, p] = 2 * D[a, b], 2 * D[b, a]
        self.A, self.B, self.M = torch.tensor(A, device=self.dev), torch.tensor(B, device=self.dev), T(M)
        L = np.polynomial.legendre.legvander(2 * x - 1, c["order"])
        self.Vi = T(np.linalg.inv(L))
        self.geometry(seed, x)
        bc, st = _box_bc(c, seed) if c["grid"] == "box" else (None, None)
        self.bc = [[None, None] for _ in range(d)]
        if bc is not None:
            for r in range(d):
                for side in range(2):
                    self.bc[r][side] = (bc[r][side], st[r][side] if st is not None else None)
        elif c["grid"] == "quad":
            self.bc = [[("supersonic-inflow", _channel_cons()), ("supersonic-outflow", None)],
                       [("slip", None), ("slip", None)]]

    def geometry(self, seed, x):
        c, d, Np = self.c, self.d, self.Np
        lo, hi = _BOX[c["flow"]]
        n = _n(c)
        if c["grid"] == "box":
            h = [(hi[r] - lo[r]) / n[r] for r in range(d)]
            self.J = math.prod(h)
            self.Ja = [[(self.J / h[r] if a == r else 0.0) for a in range(d)] for r in range(d)]
            return
        xt = torch.tensor(x, device=self.dev)

        def along(v, r):
            s = [1] * (2 * d)
            s[2 * d - 1 - r] = Np
            return v.reshape(s)
        J = [[0.0] * d for _ in range(d)]   # dx_a / dxi_b
        for bits, p in _corners(_vertices(c, seed)).items():
            P = torch.tensor(p, device=self.dev)
            for b in range(d):
                N = -1.0 if not bits[b] else 1.0
                for r in range(d):
                    if r != b:
                        N = N * along(xt if bits[r] else 1.0 - xt, r)
                for a in range(d):
                    J[a][b] = J[a][b] + N * P[..., a].reshape(tuple(reversed(n)) + (1,) * d)
        full = tuple(reversed(n)) + (Np,) * d
        J = [[(q + torch.zeros(full, device=self.dev, dtype=torch.float64)) for q in row] for row in J]
        if d == 2:
            self.Ja = [[J[1][1], -J[0][1]], [-J[1][0], J[0][0]]]
            self.J = J[0][0] * J[1][1] - J[0][1] * J[1][0]
        else:
            self.Ja = []
            for r in range(3):
                b, e = (r + 1) % 3, (r + 2) % 3
                self.Ja.append([J[(a + 1) % 3][b] * J[(a + 2) % 3][e] - J[(a + 2) % 3][b] * J[(a + 1) % 3][e]
                                for a in range(3)])
            self.J = sum(J[a][0] * self.Ja[0][a] for a in range(3))

    # node axis and element axis of direction r in [e.. , n..] arrays
    def na(self, r):
        return 2 * self.d - 1 - r

    def at(self, q, r, i):
        """Node i (an index, kept as an axis of length 1, or an index list) of direction r."""
        if not torch.is_tensor(q):
            return q
        if torch.is_tensor(i):
            return q.index_select(self.na(r), i)
        return q.narrow(self.na(r), i % self.Np, 1)

    def sums(self, mat, q, r):
        """sum_m mat[a, m] q[.. m ..] along direction r."""
        return torch.movedim(torch.tensordot(q, mat, dims=([self.na(r)], [1])), -1, self.na(r))

    def quants(self, U):
        d = self.d
        rho = U[0]
        v = [U[1 + a] / rho for a in range(d)]
        p = (GAMMA - 1.0) * (U[d + 1] - 0.5 * rho * sum(q * q for q in v))
        lam = torch.sqrt(sum(q * q for q in v)) + torch.sqrt(GAMMA * p / rho)
        return dict(rho=rho, v=v, p=p, beta=0.5 * rho / p, lam=lam, U=U)

    def pick(self, q, r, i):
        g = lambda t: self.at(t, r, i)  # noqa: E731
        return dict(rho=g(q["rho"]), v=[g(t) for t in q["v"]], p=g(q["p"]), beta=g(q["beta"]), lam=g(q["lam"]),
                    U=[g(t) for t in q["U"]])

    @staticmethod
    def logmean(x, y):
        f = (y - x) / (y + x)
        u = f * f
        series = (x + y) * 52.5 / (105.0 + u * (35.0 + u * (21.0 + u * 15.0)))
        return torch.where(u < 1e-4, series, (y - x) / torch.log(torch.where(u < 1e-4, 2.0 * x, y) / x))

    def flux(self, a, b, n, diss):
        """Chandrashekar's flux for the normal n, with its dissipation if asked."""
        d = self.d
        gm1 = GAMMA - 1.0
        rl, bl = self.logmean(a["rho"], b["rho"]), self.logmean(a["beta"], b["beta"])
        vm = [0.5 * (p + q) for p, q in zip(a["v"], b["v"])]
        Vn = sum(vm[k] * n[k] for k in range(d))
        ph = 0.5 * (a["rho"] + b["rho"]) / (a["beta"] + b["beta"])
        h = 0.5 / (bl * gm1) + ph / rl + sum(-0.25 * (p * p + q * q) + m * m for p, q, m in zip(a["v"], b["v"], vm))
        F = [rl * Vn] + [rl * Vn * vm[k] + ph * n[k] for k in range(d)] + [rl * Vn * h]
        if diss:
            nn = sum(q * q for q in n)
            nd = torch.sqrt(nn) if torch.is_tensor(nn) else math.sqrt(nn)
            hl = 0.5 * torch.maximum(a["lam"], b["lam"]) * nd
            dr, rm = b["rho"] - a["rho"], 0.5 * (a["rho"] + b["rho"])
            E = 0.5 * dr / (gm1 * bl) + 0.5 * rm / gm1 * (1.0 / b["beta"] - 1.0 / a["beta"])
            for k in range(d):
                E = E + 0.5 * dr * a["v"][k] * b["v"][k] + rm * (b["v"][k] - a["v"][k]) * vm[k]
            for k in range(d + 1):
                F[k] = F[k] - hl * (b["U"][k] - a["U"][k])
            F[d + 1] = F[d + 1] - hl * E
        return F

    def boundary(self, kind, outer, s, n):
        """The outward boundary flux of the interior face states s, and the wave speed."""
        d = self.d
        if kind == "slip":
            nd = math.sqrt(sum(q * q for q in n)) if not any(torch.is_tensor(q) for q in n) else \
                torch.sqrt(sum(q * q for q in n))
            un = sum(s["v"][k] * n[k] for k in range(d)) / nd
            a = torch.sqrt(GAMMA * s["p"] / s["rho"])
            g, g1 = GAMMA - 1.0, GAMMA + 1.0
            shock = s["p"] + 0.25 * un * g1 * s["rho"] * (
                un + torch.sqrt(un * un + 8.0 / g1 / s["rho"] * s["p"] * (g / g1 + 1.0)))
            rare = s["p"] * torch.clamp(1.0 + 0.5 * g * un / a, min=1e-4) ** (2.0 * GAMMA / g)
            ps = torch.where(un > 0, shock, rare)
            z = torch.zeros_like(ps)
            return [z] + [ps * n[k] for k in range(d)] + [z], s["lam"].max()
        if kind == "supersonic-outflow":
            o = s
        else:
            o = self.quants([torch.full_like(s["rho"], float(q)) for q in outer])
        return self.flux(s, o, n, True), torch.maximum(s["lam"], o["lam"]).max()

    def indicator(self, q):
        d, Np, c = self.d, self.Np, self.c
        m = q["rho"] * q["p"]
        for r in range(d):
            m = self.sums(self.Vi, m, r)
        e = m * m
        nodes = tuple(range(d, 2 * d))

        def low(k):
            t = e
            for r in range(d):
                t = t.narrow(self.na(r), 0, k)
            return t.sum(dim=nodes) if k > 0 else torch.zeros_like(e.sum(dim=nodes))
        mm, m1, m2 = low(Np), low(Np - 1), low(Np - 2)
        eta = torch.maximum(1.0 - m1 / mm, 1.0 - m2 / m1)
        th = 0.5 * 10.0 ** (-1.8 * c["order"] ** 0.25)
        al = 1.0 / (1.0 + torch.exp(-9.21024 * (eta - th) / th))
        al = torch.where(al < 0.001, 0.0 * al, torch.where(al > 0.999, 0.0 * al + 1.0, al))
        return torch.clamp(al, max=_alpha_max(c)).reshape(al.shape + (1,) * d)

    def viscous(self, q):
        """Volume terms [nv - 1] of the viscous flux and the face traces
        Fv . n per (direction, side)."""
        d = self.d
        nv = d + 2
        b2 = 2.0 * q["beta"]
        s = torch.log(q["p"]) - GAMMA * torch.log(q["rho"])
        W = [(GAMMA - s) / (GAMMA - 1.0) - 0.5 * b2 * sum(v * v for v in q["v"])] + [b2 * v for v in q["v"]] + [-b2]
        G = [[0.0] * nv for _ in range(d)]   # G[a][v] = d w_v / dx_a
        for v in range(1, nv):
            for r in range(d):
                s = self.sums(self.D, W[v], r)
                for a in range(d):
                    G[a][v] = G[a][v] + s * self.Ja[r][a]
            for a in range(d):
                G[a][v] = G[a][v] / self.J
            for r in range(d):
                ea, na = self.d - 1 - r, self.na(r)
                lowf, hif = self.at(W[v], r, 0), self.at(W[v], r, -1)
                jh = 0.5 * (torch.roll(lowf, -1, ea) - hif)
                jl = 0.5 * (lowf - torch.roll(hif, 1, ea))
                for a in range(d):
                    if not torch.is_tensor(self.Ja[r][a]) and self.Ja[r][a] == 0.0:
                        continue
                    for i, jump in ((self.Np - 1, jh), (0, jl)):
                        add = jump * self.at(self.Ja[r][a], r, i) / (self.w[0] * self.at(self.J, r, i))
                        G[a][v].narrow(na, i, 1).add_(add)
        # velocity and temperature (p / rho = -1 / w_last) gradients
        T = q["p"] / q["rho"]
        gv = [[T * (G[a][1 + k] + q["v"][k] * G[a][nv - 1]) for k in range(d)] for a in range(d)]
        gT = [T * T * G[a][nv - 1] for a in range(d)]
        div = sum(gv[a][a] for a in range(d))
        lam = MU * GAMMA / PR / (GAMMA - 1.0)
        F = [[None] * d for _ in range(nv - 1)]
        for a in range(d):
            for k in range(d):
                F[k][a] = MU * (gv[a][k] + gv[k][a] - (2.0 / 3.0 * div if a == k else 0.0))
            F[nv - 2][a] = sum(q["v"][k] * F[k][a] for k in range(d)) + lam * gT[a]
        vol = []
        for v in range(nv - 1):
            t = 0.0
            for r in range(d):
                t = t + self.sums(self.Dh, sum(F[v][a] * self.Ja[r][a] for a in range(d)), r)
            vol.append(t)
        tr = [[[sum(self.at(F[v][a], r, i) * self.at(self.Ja[r][a], r, i) for a in range(d)) for v in range(nv - 1)]
               for i in (0, self.Np - 1)] for r in range(d)]
        return vol, tr

    def rhs(self, U):
        d, Np, c = self.d, self.Np, self.c
        nv = d + 2
        q = self.quants([U[v] for v in range(nv)])
        lam = q["lam"].max()
        al = self.indicator(q) if c["blend"] else None
        visc, tr = self.viscous(q) if c["ns"] else (None, None)
        vol = [0.0] * nv
        fv = [0.0] * nv
        surf = [torch.zeros_like(U[0]) for _ in range(nv)]
        for r in range(d):
            na, ea = self.na(r), d - 1 - r
            n = [0.5 * (self.at(m, r, self.A) + self.at(m, r, self.B)) if torch.is_tensor(m) else m
                 for m in self.Ja[r]]
            F = self.flux(self.pick(q, r, self.A), self.pick(q, r, self.B), n, False)
            for v in range(nv):
                vol[v] = vol[v] - self.sums(self.M, F[v], r)
            del F
            if c["blend"]:
                n = []
                for m in self.Ja[r]:
                    if not torch.is_tensor(m):
                        n.append(m)
                        continue
                    dm = self.sums(self.D, m, r)
                    k, parts = self.at(m, r, 0), []
                    for i in range(Np - 1):
                        k = k + self.w[i] * self.at(dm, r, i)
                        parts.append(k)
                    n.append(torch.cat(parts, na))
                i = torch.arange(Np - 1, device=self.dev)
                G = self.flux(self.pick(q, r, i), self.pick(q, r, i + 1), n, True)
                for v in range(nv):
                    z = torch.zeros_like(G[v].narrow(na, 0, 1))
                    ext = torch.cat([z, G[v], z], na)
                    shape = [1] * (2 * d)
                    shape[na] = Np
                    wt = torch.tensor(self.w, device=self.dev).reshape(shape)
                    fv[v] = fv[v] + (ext.narrow(na, 0, Np) - ext.narrow(na, 1, Np)) / (self.J * wt)
                del G
            lo, hi = self.pick(q, r, 0), self.pick(q, r, -1)
            roll = lambda t, k: torch.roll(t, k, ea)  # noqa: E731
            nxt = dict(rho=roll(lo["rho"], -1), v=[roll(t, -1) for t in lo["v"]], p=roll(lo["p"], -1),
                       beta=roll(lo["beta"], -1), lam=roll(lo["lam"], -1), U=[roll(t, -1) for t in lo["U"]])
            nh = [self.at(m, r, -1) for m in self.Ja[r]]
            nl = [self.at(m, r, 0) for m in self.Ja[r]]
            F = self.flux(hi, nxt, nh, True)     # the face above each element
            if c["ns"]:
                for v in range(nv - 1):
                    F[1 + v] = F[1 + v] - 0.5 * (tr[r][1][v] + roll(tr[r][0][v], -1))
            H = [-f for f in F]
            Lw = [roll(f, 1) for f in F]
            if self.bc[r][0] is not None:
                first = lambda t: t.narrow(ea, 0, 1) if torch.is_tensor(t) else t  # noqa: E731
                last = lambda t: t.narrow(ea, t.shape[ea] - 1, 1) if torch.is_tensor(t) else t  # noqa: E731
                for side, end, s, nn, dst in ((0, first, lo, [-m for m in nl], Lw), (1, last, hi, nh, H)):
                    kind, outer = self.bc[r][side]
                    sb = dict(rho=end(s["rho"]), v=[end(t) for t in s["v"]], p=end(s["p"]), beta=end(s["beta"]),
                              lam=end(s["lam"]), U=[end(t) for t in s["U"]])
                    Fb, lb = self.boundary(kind, outer, sb, [end(m) for m in nn])
                    lam = torch.maximum(lam, lb)
                    for v in range(nv):
                        dst[v] = dst[v].clone()
                        end(dst[v]).copy_(-Fb[v])
            for v in range(nv):
                surf[v].narrow(na, Np - 1, 1).add_(H[v] / (self.w[0] * self.at(self.J, r, -1)))
                surf[v].narrow(na, 0, 1).add_(Lw[v] / (self.w[0] * self.at(self.J, r, 0)))
        out = []
        for v in range(nv):
            t = vol[v] * (1.0 - al) if al is not None else vol[v]
            if c["ns"] and v > 0:
                t = t + visc[v - 1]
            t = t / self.J
            if al is not None:
                t = t + al * fv[v]
            out.append(t + surf[v])
        return torch.stack(out), float(lam)

    def step(self, u, dt):
        f, l0 = self.rhs(u)
        y = u + dt * f
        f, l1 = self.rhs(y)
        y = 0.75 * u + 0.25 * (y + dt * f)
        f, l2 = self.rhs(y)
        return u / 3.0 + 2.0 / 3.0 * (y + dt * f), max(l0, l1, l2)


def exact(case, seed):
    c = case
    if c["grid"] == "ensemble":
        out = []
        for m, sd in _members(c, seed):
            u, S = _state(m, sd), _Scheme(m, sd)
            for _ in range(c["steps"]):
                u, _l = S.step(u, _dt(m))
            out.append(u.reshape(-1))
        return out
    u, S = _state(c, seed), _Scheme(c, seed)
    if c["entry"] == "mult":
        return S.rhs(u)[0].reshape(-1)
    if c["entry"] == "step":
        for _ in range(c["steps"]):
            u, _l = S.step(u, _dt(c))
        return u.reshape(-1)
    t, lam = 0.0, S.rhs(u)[1]
    for _ in range(c["steps"]):
        dt = 0.5 * _hmin(c) / (lam * (c["order"] + 1) ** 2)
        u, l1 = S.step(u, dt)
        lam = max(lam, l1)
        t += dt
    return {"u": u.reshape(-1), "t": t, "n": c["steps"]}
