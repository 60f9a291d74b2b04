"""Inputs at the edge of what the operators take, against the FP64 oracle:
negative densities and pressures whose fluxes are finite, and mesh sizes far
from 1."""
import numpy as np
import pytest

import oracle_lib as O
import quad_meshes as Q
from prandtl_amd import DGSEMOperator, cases
from prandtl_amd.operator import HexMesh

pytestmark = pytest.mark.gpu

TOL = 1e-12   # the repository's parity bar


def mult(op, u, dev):
    import torch
    du = torch.tensor(np.ascontiguousarray(u).reshape(-1), dtype=torch.float64, device=dev)
    out = torch.empty_like(du)
    op.Mult(du, out)
    torch.cuda.synchronize()
    return out.cpu().numpy()


def rel_max(a, b):
    return float(np.abs(a - b).max() / np.abs(b).max())


# (density, pressure) signs with real wave speeds; without dissipation also a
# negative pressure alone
SIGNS = [(-1.0, -2.0, False), (-1.0, -2.0, True), (1.0, -2.0, True)]


@pytest.mark.parametrize("equal", [True, False])
@pytest.mark.parametrize("rho0,p0,ec", SIGNS)
@pytest.mark.parametrize("dim,order,n", [(2, 3, 4), (2, 4, 70), (3, 2, 4), (3, 3, 3), (3, 4, 9), (3, 6, 3)])
def test_negative_values(cuda, dim, order, n, rho0, p0, ec, equal):
    """The mean of two equal negative values is the value, also where they differ
    in their last bits (rho/(2p) of a constant ratio, at a power of two); of
    different ones of the same sign it is their logarithmic mean."""
    cfg = dict(dim=dim, order=order, nelem=(n, n + 1, n)[:dim], lo=(0.0,) * dim, hi=(1.0,) * dim, quirks=False,
               ec_surface=ec)
    op, orc = DGSEMOperator(**cfg), O.Oracle(threads=16, **cfg)
    rng = np.random.default_rng(dim * 10 + order)
    shape = (orc.NE, orc.K)
    wave = 1.0 if equal else 1.0 + 0.8 * rng.random(shape)
    rho = np.full(shape, rho0) * wave
    p = np.full(shape, p0) * (1.0 + 0.2 * rng.random(shape) if rho0 < 0 else wave)
    v = [0.3 + 0.2 * rng.random(shape) for _ in range(dim)]
    u = np.stack([rho] + [rho * x for x in v] + [p / 0.4 + 0.5 * rho * sum(x * x for x in v)])
    out, ref = mult(op, u, cuda), orc.Mult(u)
    assert np.isfinite(ref).all()
    assert np.isfinite(out).all()
    r = rel_max(out, ref)
    print("%dD N=%d %g %g ec=%d equal=%d: %.2e" % (dim, order, rho0, p0, ec, equal, r), flush=True)
    assert r <= TOL


@pytest.mark.parametrize("size", [1e-80, 1.0, 1e80])
@pytest.mark.parametrize("order,n", [(2, 3), (3, 3), (3, 11), (4, 3)])
def test_mesh_size(cuda, order, n, size):
    """Hexahedra whose normals' squares are out of range: the normals are squares
    of lengths, the right-hand side (of an Euler state) is a rate per length."""
    d = Q.hex_grid(n, 3, n, (0.0,) * 3, (size, 0.8 * size, 0.6 * size), periodic=(False, True, True), perturb=0.2, seed=1)
    d.update(attr_bc=["slip", "symmetry"], attr_state=[(0.0,) * 5] * 2)
    mesh = HexMesh(d["vert"], d["elem"], d["bdr"], d["bdr_attr"], d["elem_coords"])
    kw = dict(blending=True, quirks=False)
    op = DGSEMOperator.hex(mesh, order, bc={1: "slip", 2: "symmetry"}, **kw)
    orc = O.Oracle.hex(d, order, threads=16, **kw)
    u = cases.random_smooth_state(orc.coords() / size, 3, 3, L=[1.0, 0.8, 0.6])
    out, ref = mult(op, u, cuda), orc.Mult(u)
    assert np.isfinite(ref).all()
    r = rel_max(out, ref)
    print("N=%d %d size %g: %.2e" % (order, n, size, r), flush=True)
    assert r <= TOL
