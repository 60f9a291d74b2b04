"""Boundary sides of quadrilateral and hexahedral meshes: every type, on every
local face (elements renumbered, their frames turned), for each order and each
of the kernels that a mesh's size selects, against the FP64 oracle.

Bar: the metrics' rounding, eps L / h, magnified by the derivative at most
N (N + 1) / 2 times relative to the sides' jumps: 2.2e-16 * 81 * 15 = 2.7e-13 on
the finest mesh here, against the repository's 1e-12.
"""
import numpy as np
import pytest

import oracle_lib as O
import quad_meshes as Q
from prandtl_amd import DGSEMOperator, cases
from prandtl_amd.operator import HexMesh, QuadMesh

pytestmark = pytest.mark.gpu

TOL = 1e-12
G = 1.4
FORMS = {"euler": dict(quirks=False), "ns": dict(parabolic=True, mu=0.001, Pr=0.71, quirks=False),
         "faithful": dict(parabolic=True, mu=0.001, Pr=0.71, quirks=True)}
QUAD = {1: [(7, 6), (80, 81)], 2: [(7, 6), (75, 74)], 3: [(7, 6), (66, 67)], 4: [(7, 6), (58, 57)], 5: [(7, 6), (50, 49)]}
HEX = {2: [(3, 3, 4), (24, 24, 25)], 3: [(3, 3, 4), (9, 10, 10), (11, 10, 10)], 4: [(3, 3, 4), (7, 8, 7), (10, 9, 9)]}
IN, OUT, SLIP, SYM, SPEC, WALL = ("supersonic-inflow", "supersonic-outflow", "slip", "symmetry", "specified-state",
                                  "no-slip-adiabatic")
EULER_SIDES = {"a": (IN, OUT, SLIP, SYM, SPEC, SLIP), "b": (SLIP, SYM, SPEC, SLIP, IN, OUT), "c": (SYM, SLIP, IN, OUT, SLIP, SYM)}
NS_SIDES = {"a": (IN, OUT, WALL, WALL, SPEC, WALL), "b": (WALL, WALL, IN, OUT, WALL, SPEC)}


def cons(rho, v, p):
    v = np.asarray(v, float)
    return np.array([rho, *(rho * v), p / (G - 1) + 0.5 * rho * np.dot(v, v)])


def run(dev, dim, order, n, form, sides):
    import torch
    if dim == 2:
        d, _ = Q.relabel(Q.grid(*n, periodic=(False, False), perturb=0.2, seed=8))
    else:
        d = Q.hex_relabel(Q.hex_grid(*n, periodic=(False,) * 3, perturb=0.2, seed=8))[0]
    kinds = list((NS_SIDES if form != "euler" else EULER_SIDES)[sides][:2 * dim])
    flow = cons(1.3, [1.9, 0.3, -0.2][:dim], 1.0)
    wall = np.zeros(dim + 2)
    wall[:dim] = [0.2, -0.1, 0.3][:dim]
    states = [wall if k == WALL else flow for k in kinds]
    d.update(attr_bc=kinds, attr_state=[np.concatenate([s, np.zeros(5)])[:4 if dim == 2 else 5] for s in states])
    kw = dict(FORMS[form], blending=order == 3)
    bc = {i + 1: (k, s) for i, (k, s) in enumerate(zip(kinds, states))}
    if dim == 2:
        op = DGSEMOperator.quad(QuadMesh(d["vert"], d["elem"], d["bdr"], d["bdr_attr"]), order, bc=bc, **kw)
        orc = O.Oracle.quad(d, order, threads=16, **kw)
    else:
        op = DGSEMOperator.hex(HexMesh(d["vert"], d["elem"], d["bdr"], d["bdr_attr"]), order, bc=bc, **kw)
        orc = O.Oracle.hex(d, order, threads=16, **kw)
    u = cases.random_smooth_state(orc.coords(), dim, 9, L=[1.0] * dim)
    du = torch.tensor(np.ascontiguousarray(u).reshape(-1), dtype=torch.float64, device=dev)
    out = torch.empty_like(du)
    op.Mult(du, out)
    torch.cuda.synchronize()
    ref = orc.Mult(u)
    r = np.abs(out.cpu().numpy() - ref).max() / np.abs(ref).max()
    print("%dD N=%d %s %s %s: %.2e" % (dim, order, n, form, sides, r), flush=True)
    assert r <= TOL


CASES = [(f, s) for f in FORMS for s in (EULER_SIDES if f == "euler" else NS_SIDES)]


@pytest.mark.parametrize("form,sides", CASES)
@pytest.mark.parametrize("order,n", [(N, n) for N in QUAD for n in QUAD[N]])
def test_quads(cuda, order, n, form, sides):
    run(cuda, 2, order, n, form, sides)


@pytest.mark.parametrize("form,sides", CASES)
@pytest.mark.parametrize("order,n", [(N, n) for N in HEX for n in HEX[N]])
def test_hexahedra(cuda, order, n, form, sides):
    run(cuda, 3, order, n, form, sides)
