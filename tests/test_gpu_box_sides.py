"""Boundary sides of boxes: every type on every side, for each order and each
of the kernels that a mesh's size selects.

The meshes of an order lie below and above the element counts at which the
right-hand side changes from node threads to line threads and from the small
workgroup to the natural one.  Against the FP64 oracle at the repository's
parity bar.
"""
import numpy as np
import pytest

import oracle_lib as O
from prandtl_amd import DGSEMOperator, cases

pytestmark = pytest.mark.gpu

TOL = 1e-12
G = 1.4
NS = dict(parabolic=True, mu=0.02, Pr=0.71)

# 3-D: node threads up to 341, 256 and 232 elements at N = 3, 4, 5 (faithful
# Navier-Stokes 768 and 554 at N = 3, 4; N = 2 only with blending), the small
# workgroup up to 1023, 767 and 511, at N = 2 up to 13,824; 2-D: node threads up
# to 6,144, 5,376, 4,096 and 2,496 elements at most
SIZES = {2: {2: [(5, 4), (90, 91)], 3: [(5, 4), (80, 81)], 4: [(5, 4), (66, 67)], 5: [(5, 4), (61, 60)]},
         3: {2: [(3, 4, 5), (9, 9, 8), (24, 24, 25)], 3: [(3, 4, 5), (8, 8, 7), (11, 10, 10)],
             4: [(3, 4, 5), (7, 8, 7), (10, 9, 9)], 5: [(3, 4, 5), (7, 7, 7), (9, 8, 8)],
             6: [(3, 4, 3)], 7: [(3, 2, 3)]}}
MESHES = [(d, n, s) for d in SIZES for n in SIZES[d] for s in SIZES[d][n]]


def cons(rho, v, p):
    v = np.asarray(v, float)
    return np.array([rho, *(rho * v), p / (G - 1) + 0.5 * rho * np.dot(v, v)])


def sides(dim, kind):
    """All sides of one type, or inflow and outflow in turn."""
    st = cons(1.3, [2.1, 0.4, -0.3][:dim], 1.0)
    kinds = ("supersonic-inflow", "supersonic-outflow") if kind == "in-out" else (kind, kind)
    bc = [kinds if r % 2 == 0 else kinds[::-1] for r in range(dim)]
    wall = np.array([0.3, -0.2, 0.1, 0.0, 0.0])
    wall[dim:] = 0.0
    state = wall[:dim + 2] if kind == "no-slip-adiabatic" else st
    return dict(bc=bc, bc_state=[(state, state)] * dim)


def check(dev, cfg, seed):
    import torch
    op, orc = DGSEMOperator(**cfg), O.Oracle(threads=16, **cfg)
    X = cases.node_coords(cfg["dim"], cfg["order"], cfg["nelem"], cfg["lo"], cfg["hi"])
    u = cases.random_smooth_state(X, cfg["dim"], seed, L=[h - l for l, h in zip(cfg["lo"], cfg["hi"])])
    du = torch.tensor(u.reshape(-1), dtype=torch.float64, device=dev)
    out = torch.empty_like(du)
    op.Mult(du, out)
    torch.cuda.synchronize()
    ref = orc.Mult(u)
    return np.abs(out.cpu().numpy() - ref).max() / np.abs(ref).max()


def box(dim, order, nelem, **kw):
    return dict(dim=dim, order=order, nelem=nelem, lo=(0.0,) * dim, hi=(1.0, 1.1, 0.9)[:dim], quirks=False, **kw)


@pytest.mark.parametrize("blend", [False, True])
@pytest.mark.parametrize("kind", ["slip", "symmetry", "specified-state", "in-out"])
@pytest.mark.parametrize("dim,order,nelem", MESHES)
def test_box_sides(cuda, dim, order, nelem, kind, blend):
    cfg = box(dim, order, nelem, blending=blend, **sides(dim, kind))
    r = check(cuda, cfg, 11)
    print("%dD N=%d %s %s blend=%d: %.2e" % (dim, order, nelem, kind, blend, r), flush=True)
    assert r <= TOL


@pytest.mark.parametrize("quirks", [False, True])
@pytest.mark.parametrize("dim,order,nelem", MESHES)
def test_box_no_slip_sides(cuda, dim, order, nelem, quirks):
    cfg = dict(box(dim, order, nelem, **NS, **sides(dim, "no-slip-adiabatic")), quirks=quirks)
    r = check(cuda, cfg, 12)
    print("%dD N=%d %s no-slip quirks=%d: %.2e" % (dim, order, nelem, quirks, r), flush=True)
    assert r <= TOL


@pytest.mark.parametrize("order", range(2, 8))
@pytest.mark.parametrize("wall", range(3))
def test_tangential_stream_along_walls(cuda, order, wall):
    """A uniform stream along two slip walls is steady: the wall pressure is
    the stream's."""
    import torch
    bc = [("periodic", "periodic")] * 3
    bc[wall] = ("slip", "slip")
    for nelem in SIZES[3][order]:
        op = DGSEMOperator(dim=3, order=order, nelem=nelem, lo=(0.0,) * 3, hi=(2.0,) * 3, quirks=False, bc=bc)
        for vel in np.eye(3):
            vel = np.where(np.arange(3) == wall, 0.0, vel + 0.25)
            u = np.zeros((5, op.NE, op.K))
            u += cons(1.0, vel, 7.0)[:, None, None]
            du = torch.tensor(u.reshape(-1), dtype=torch.float64, device=cuda)
            out = torch.empty_like(du)
            op.Mult(du, out)
            # relative to the wall pressure's own term p / (w_0 h)
            scale = 7.0 * order * (order + 1) * max(nelem) / 2.0
            r = float(out.abs().max()) / scale
            print("N=%d wall %d %s: %.2e" % (order, wall, nelem, r), flush=True)
            assert r <= 1e-13
