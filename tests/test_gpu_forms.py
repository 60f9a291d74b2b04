"""Every form of the equations (Euler, corrected, faithful and mixed Navier-Stokes,
axisymmetric) in each of the kernels that a mesh's size selects: node threads,
line threads in the small workgroup, line threads in the natural one.

Bit for bit between the kernels, where a box repeats along x: its elements see
the same neighbours as in one period.  And against the FP64 oracle at the
repository's parity bar, on meshes below and above the element counts at which
the kernel changes, in the forms whose right-hand side does not cancel on fine
meshes.
"""
import numpy as np
import pytest

import oracle_lib as O
import quad_meshes as Q
from prandtl_amd import DGSEMOperator, cases
from prandtl_amd.operator import HexMesh, QuadMesh

pytestmark = pytest.mark.gpu

TOL = 1e-12
NS = dict(parabolic=True, mu=0.02, Pr=0.71)
FORMS = {"euler": dict(quirks=False), "ns": dict(NS, quirks=False), "faithful": dict(NS, quirks=True),
         "mixed": dict(NS, quirks=False, precision="mixed")}
# one mesh for each kernel of an order (3-D N = 6, 7: one kernel)
BOX2 = {2: [(7, 5), (90, 91)], 3: [(7, 5), (80, 81)], 4: [(7, 5), (66, 67)], 5: [(7, 5), (61, 60)]}
BOX3 = {2: [(3, 4, 5), (24, 24, 25)], 3: [(3, 4, 5), (8, 9, 8), (11, 10, 10)], 4: [(3, 4, 5), (8, 9, 9), (10, 9, 9)],
        5: [(3, 4, 5), (7, 7, 7), (9, 8, 8)], 6: [(3, 4, 3)], 7: [(3, 2, 3)]}
QUAD = {1: [(7, 6), (80, 81)], 2: [(7, 6), (75, 74)], 3: [(7, 6), (66, 67)], 4: [(7, 6), (58, 57)], 5: [(7, 6), (50, 49)]}
AXI = {1: [(7, 6), (130, 121)], 2: [(7, 6), (110, 101)], 3: [(7, 6), (90, 81)], 4: [(7, 6), (76, 65)], 5: [(7, 6), (65, 56)]}
HEX = {2: [(3, 3, 4), (22, 22, 23)], 3: [(3, 3, 4), (9, 10, 10), (11, 10, 10)], 4: [(3, 3, 4), (7, 8, 7), (10, 9, 9)]}
every = lambda d: [(n, s) for n in d for s in d[n]]


def mult(op, u, dev):
    import torch
    du = torch.tensor(np.ascontiguousarray(u).reshape(-1), dtype=torch.float64, device=dev)
    out = torch.empty_like(du)
    op.Mult(du, out)
    torch.cuda.synchronize()
    return out.cpu().numpy()


def check(out, ref, what):
    r = np.abs(out - ref).max() / np.abs(ref).max()
    print("%s: %.2e" % (what, r), flush=True)
    assert r <= TOL, what


@pytest.mark.parametrize("blend", [False, True])
@pytest.mark.parametrize("form", ["euler", "faithful"])
@pytest.mark.parametrize("order,nelem", every(BOX2) + every(BOX3))
def test_boxes(cuda, order, nelem, form, blend):
    dim = len(nelem)
    cfg = dict(FORMS[form], dim=dim, order=order, nelem=nelem, lo=(0.0,) * dim, hi=(1.0, 1.1, 0.9)[:dim], blending=blend)
    op, orc = DGSEMOperator(**cfg), O.Oracle(threads=16, **cfg)
    X = cases.node_coords(dim, order, nelem, cfg["lo"], cfg["hi"])
    u = cases.random_smooth_state(X, dim, 21, L=list(cfg["hi"]))
    check(mult(op, u, cuda), orc.Mult(u), "N=%d %s %s blend=%d" % (order, nelem, form, blend))


@pytest.mark.parametrize("order,n", every(QUAD))
def test_faithful_quads(cuda, order, n):
    d = Q.grid(*n, periodic=(False, True), perturb=0.2, seed=5)
    d.update(attr_bc=["supersonic-outflow"] * 2, attr_state=[(0.0,) * 4] * 2)
    kw = FORMS["faithful"]
    op = DGSEMOperator.quad(QuadMesh(d["vert"], d["elem"], d["bdr"], d["bdr_attr"], d["elem_coords"]), order,
                            bc={1: "supersonic-outflow", 2: "supersonic-outflow"}, blending=order % 2 == 0, **kw)
    orc = O.Oracle.quad(d, order, threads=16, blending=order % 2 == 0, **kw)
    u = cases.random_smooth_state(orc.coords(), 2, 22, L=[1.0, 1.0])
    check(mult(op, u, cuda), orc.Mult(u), "quads N=%d %s" % (order, n))


@pytest.mark.parametrize("blend", [False, True])
@pytest.mark.parametrize("order,n", every(AXI))
def test_axisymmetric(cuda, order, n, blend):
    d = Q.grid(*n, (0.0, 0.0), (2.0, 1.0), periodic=(False, False), perturb=0.2, seed=order)
    kinds = ["supersonic-inflow", "supersonic-outflow", "axis", "slip"]
    d.update(attr_bc=kinds, attr_state=[cases.RAMP_STATE] * 4)
    kw = dict(blending=blend, alpha_max=0.5, axisymmetric=True)
    op = DGSEMOperator.quad(QuadMesh(d["vert"], d["elem"], d["bdr"], d["bdr_attr"]), order,
                            bc={i + 1: (k, cases.RAMP_STATE) for i, k in enumerate(kinds)}, **kw)
    orc = O.Oracle.quad(d, order, threads=16, quirks=False, **kw)
    X = orc.coords()
    u = cases.axisymmetric_state(cases.random_smooth_state(X / np.array([2.0, 1.0])[:, None, None], 2, 23, amp=0.15, L=[1.0, 1.0]), X)
    out, ref = mult(op, u, cuda), orc.Mult(u)
    check(out, ref, "axisymmetric N=%d %s blend=%d" % (order, n, blend))
    lam = orc.GetMaxCharSpeed()
    assert abs(op.GetMaxCharSpeed() - lam) <= 1e-13 * lam


@pytest.mark.parametrize("form", ["euler", "ns", "faithful"])
@pytest.mark.parametrize("order,n", every(HEX))
def test_hexahedra(cuda, order, n, form):
    d = Q.hex_grid(*n, periodic=(True, True, False), perturb=0.2, seed=6)
    bc = {5: "supersonic-outflow", 6: "supersonic-outflow"}
    d.update(attr_bc=["slip"] * 4 + ["supersonic-outflow"] * 2, attr_state=[(0.0,) * 5] * 6)
    kw = FORMS[form]
    blend = order == 3
    op = DGSEMOperator.hex(HexMesh(d["vert"], d["elem"], d["bdr"], d["bdr_attr"], d["elem_coords"]), order, bc=bc,
                           blending=blend, **kw)
    orc = O.Oracle.hex(d, order, threads=16, blending=blend, **kw)
    u = cases.random_smooth_state(orc.coords(), 3, 24, L=[1.0, 1.0, 1.0])
    check(mult(op, u, cuda), orc.Mult(u), "hexahedra N=%d %s %s" % (order, n, form))


# (order, one period, its repetitions along x): the period by node threads, the
# whole by line threads
REPEAT = [(2, (8, 4), 256), (3, (8, 4), 160), (4, (8, 4), 128), (5, (8, 4), 96), (2, (2, 4, 2), 128), (2, (2, 4, 2), 1024), (3, (2, 4, 2), 64),
          (4, (2, 4, 2), 64), (5, (2, 4, 2), 32)]


@pytest.mark.parametrize("walls", [False, True])
@pytest.mark.parametrize("blend", [False, True])
@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("order,period,rep", REPEAT)
def test_repeated_period_bitwise(cuda, order, period, rep, form, blend, walls):
    dim = len(period)
    wall = "slip" if form == "euler" else "no-slip-adiabatic"
    bc = [("periodic", "periodic")] + [(wall, wall)] * (dim - 1) if walls else None
    st = [((0.0,) * (dim + 2),) * 2] * dim if walls else None
    size = lambda k: dict(nelem=(period[0] * k,) + period[1:], hi=(1.0 * k,) + (1.0,) * (dim - 1))
    kw = dict(FORMS[form], dim=dim, order=order, lo=(0.0,) * dim, blending=blend, bc=bc, bc_state=st)
    a, b = DGSEMOperator(**kw, **size(1)), DGSEMOperator(**kw, **size(rep))
    X = cases.node_coords(dim, order, period, kw["lo"], size(1)["hi"])
    u = cases.random_smooth_state(X, dim, 25, amp=0.02, L=[1.0] * dim)
    # elements with jumps of 1.5 and of 4 beside smooth ones
    jump = (np.arange(u.shape[2]) % (order + 1) > order // 2)[None, :] * np.array([0.0, 0.5, 3.0])[np.arange(u.shape[1]) % 3][:, None]
    u = u * (1.0 + jump)[None]
    nv, K = u.shape[0], u.shape[2]
    rows = u.reshape(nv, -1, period[0], K)
    big = np.tile(rows, (1, 1, rep, 1)).reshape(nv, -1, K)
    out = mult(a, u, cuda).reshape(nv, -1, period[0], K)
    all_ = mult(b, big, cuda).reshape(nv, -1, rep, period[0], K)
    assert np.isfinite(out).all()
    assert (all_ == out[:, :, None]).all()
