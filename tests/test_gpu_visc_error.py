"""Rounding of the viscous line kernel: the FP64 right-hand side of corrected
Navier-Stokes on boxes, in the relative L2 norm against the extended-precision
oracle, is no further off than the FP64 oracle's own, which sums over plain rows
of D (a quarter for the states' sampling), where the viscous terms' cancellation
dominates: fine meshes, every order."""
import numpy as np
import pytest

import oracle_lib as O
from prandtl_amd import DGSEMOperator, cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("walls", [False, True])
@pytest.mark.parametrize("order,nelem", [(2, (70, 71)), (3, (60, 61)), (4, (50, 51)), (5, (45, 44)), (2, (16, 15, 17)), (2, (24, 24, 25)),
                                         (3, (11, 12, 10)), (4, (9, 10, 9)), (5, (8, 8, 9)), (6, (6, 5, 6)), (7, (5, 4, 5))])
def test_viscous_error(cuda, order, nelem, walls):
    import torch
    dim = len(nelem)
    wall = "no-slip-adiabatic"
    cfg = dict(dim=dim, order=order, nelem=nelem, lo=(0.0,) * dim, hi=(1.0,) * dim, parabolic=True, mu=0.02, Pr=0.71,
               quirks=False, bc=[(wall, wall)] + [("periodic", "periodic")] * (dim - 1) if walls else None,
               bc_state=[((0.0,) * (dim + 2),) * 2] * dim if walls else None)
    op, orc = DGSEMOperator(**cfg), O.Oracle(threads=16, **cfg)
    X = cases.node_coords(dim, order, nelem, cfg["lo"], cfg["hi"])
    u = cases.random_smooth_state(X, dim, 31, L=[1.0] * dim)
    du = torch.tensor(u.reshape(-1), dtype=torch.float64, device=cuda)
    out = torch.empty_like(du)
    op.Mult(du, out)
    torch.cuda.synchronize()
    ext, ref = orc.Mult_extended(u), orc.Mult(u)
    e_gpu, e_orc = (np.linalg.norm(x - ext) / np.linalg.norm(ext) for x in (out.cpu().numpy(), ref))
    print("%dD N=%d walls=%d: GPU %.2e, oracle %.2e (%.2f)" % (dim, order, walls, e_gpu, e_orc, e_gpu / e_orc), flush=True)
    assert e_gpu <= 1.25 * e_orc
