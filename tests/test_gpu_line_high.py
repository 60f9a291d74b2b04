"""The high-order line kernel (3-D boxes of order 5..7) against the oracle:
element counts its elements per workgroup do not divide, blended and
unblended, Navier-Stokes in both modes and the mixed form, boundary sides;
and the launch shapes of order 5.  The bar is the repository's parity bar
(1e-12 relative max-norm; states where the FP64 oracle itself is further than
that from its extended-precision form: within twice its distance)."""
import math

import numpy as np
import pytest

import oracle_lib as O
from prandtl_amd import DGSEMOperator, cases

pytestmark = pytest.mark.gpu

TWO_PI = 2.0 * math.pi
NS = dict(parabolic=True, mu=0.01, Pr=0.71)
WALL = ("no-slip-adiabatic", "no-slip-adiabatic")
PER = ("periodic", "periodic")
KINDS = {
    "euler": dict(quirks=False),
    "euler_ec": dict(quirks=False, ec_surface=True),
    "blend": dict(quirks=True, blending=True, alpha_max=0.5),
    "blend_full": dict(quirks=False, blending=True, alpha_max=1.0),
    "ns": dict(quirks=False, **NS),
    "ns_faithful_blend": dict(quirks=True, blending=True, alpha_max=0.1, **NS),
    "slip": dict(quirks=False, bc=[("slip", "slip"), ("symmetry", "slip"), PER]),
    "ns_walls_blend": dict(quirks=False, blending=True, alpha_max=0.5, bc=[PER, WALL, PER],
                           bc_state=[(None, None), ((0.1, 0.0, 0.2, 0.05, 0.0), (0.0,) * 5), (None, None)], **NS),
    "ns_faithful_walls": dict(quirks=True, bc=[PER, WALL, PER],
                              bc_state=[(None, None), ((0.0,) * 5, (0.0,) * 5), (None, None)], **NS),
}


def rel(a, b):
    return float(np.abs(a - b).max() / np.abs(b).max())


@pytest.mark.parametrize("N,nelem", [(5, (3, 3, 3)), (6, (2, 2, 3)), (7, (3, 2, 2))])
@pytest.mark.parametrize("kind", sorted(KINDS))
def test_high_order_parity(cuda, N, nelem, kind):
    import torch
    cfg = dict(dim=3, order=N, nelem=nelem, lo=(0.0,) * 3, hi=(TWO_PI, 2.0, 3.0), **KINDS[kind])
    op, orc = DGSEMOperator(**cfg), O.Oracle(threads=8, **cfg)
    X = cases.node_coords(3, N, nelem, cfg["lo"], cfg["hi"])
    u = cases.random_smooth_state(X, 3, 29, amp=0.2, L=list(cfg["hi"]))
    if cfg.get("blending"):
        # jumps inside some elements, so that some blend and some do not
        step = (np.arange(u.shape[1]) % 3 == 0)[:, None] & (np.arange(u.shape[2]) % (N + 1) > N // 2)[None, :]
        u = u * (1.0 + 0.4 * step)[None]
    du = torch.tensor(u.reshape(-1), dtype=torch.float64, device=cuda)
    out = torch.empty_like(du)
    op.Mult(du, out)
    torch.cuda.synchronize()
    ref = orc.Mult(u)
    r = rel(out.cpu().numpy(), ref)
    print("high order %s N=%d: %.3e" % (kind, N, r), flush=True)
    if r > 1e-12:
        ext = orc.Mult_extended(u)
        e_orc = rel(ref, ext)
        assert e_orc > 1e-12 and rel(out.cpu().numpy(), ext) <= 2.0 * e_orc
    if cfg.get("blending"):
        al, eta = op.alpha()
        assert np.abs(eta - orc.eta()).max() <= 1e-12 and np.abs(al - orc.alpha()).max() <= 1e-10
        assert (al > 0).sum() > 0
    if not (cfg.get("parabolic") and cfg["quirks"]):
        # (the faithful Navier-Stokes oracle also counts the aliased face states' speeds)
        lam = orc.GetMaxCharSpeed()
        assert abs(op.GetMaxCharSpeed() - lam) <= 1e-14 * lam
    op.Step(du, 1e-4)
    torch.cuda.synchronize()
    assert rel(du.cpu().numpy(), orc.Step(u.reshape(-1).copy(), 1e-4)) <= 1e-12


@pytest.mark.parametrize("blend", [False, True])
def test_high_order_shapes(cuda, blend):
    import torch
    cfg = dict(dim=3, order=5, nelem=(3, 3, 3), lo=(0.0,) * 3, hi=(1.0, 2.0, 3.0), quirks=False, blending=blend)
    op = DGSEMOperator(**cfg)
    X = cases.node_coords(3, 5, cfg["nelem"], cfg["lo"], cfg["hi"])
    u = cases.random_smooth_state(X, 3, 31, amp=0.5, L=list(cfg["hi"]))
    u = u * (1.0 + 0.3 * (np.arange(u.shape[1]) % 2))[None, :, None]
    du = torch.tensor(u.reshape(-1), dtype=torch.float64, device=cuda)
    a, b = torch.empty_like(du), torch.empty_like(du)
    op.Mult(du, a)
    op.set_shape("rhs", 3)
    op.Mult(du, b)
    torch.cuda.synchronize()
    assert torch.equal(a, b)
