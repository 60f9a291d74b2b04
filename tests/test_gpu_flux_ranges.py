"""The two-point flux over the ranges of its logarithmic means.

The kernels evaluate log means by a short series (neighbouring values within
2%), a polynomial (up to a ratio of 2) or the logarithm (beyond).  States
whose nodes differ by ratios on both sides of each limit, element kernels of
every kind, against the FP64 oracle.  The bar is the repository's parity bar:
node-wise random states leave no cancellation in the RHS, and the oracle's own
log mean is good to 5e-15 (its quotient (y-x)/log(y/x) just above 2%).
"""
import numpy as np
import pytest

import oracle_lib as O
from prandtl_amd import DGSEMOperator, cases

pytestmark = pytest.mark.gpu

BOX = {
    "2d": dict(dim=2, order=3, nelem=(4, 5), lo=(-1.0, -1.0), hi=(1.0, 1.0)),
    "2d_n5_blend": dict(dim=2, order=5, nelem=(3, 3), lo=(-1.0, -1.0), hi=(1.0, 1.0), blending=True),
    "3d_n3": dict(dim=3, order=3, nelem=(3, 2, 4), lo=(0.0,) * 3, hi=(1.0, 2.0, 3.0), quirks=False),
    "3d_n4_tile": dict(dim=3, order=4, nelem=(2, 2, 3), lo=(0.0,) * 3, hi=(1.0, 2.0, 3.0), quirks=False),
    "3d_n6": dict(dim=3, order=6, nelem=(2, 2, 2), lo=(0.0,) * 3, hi=(1.0, 2.0, 3.0), quirks=False),
    "3d_slip": dict(dim=3, order=3, nelem=(2, 2, 3), lo=(0.0,) * 3, hi=(1.0, 2.0, 3.0), quirks=False,
                    bc=[("slip", "slip"), ("slip", "slip"), ("periodic", "periodic")]),
}


# ratios inside, around (u = 1e-4 at 1.0202, u = 1/9 at 2) and beyond the limits
@pytest.mark.parametrize("ratio", [1.0, 1.0 + 1e-9, 1.02, 1.0205, 1.3, 1.999, 2.001, 30.0])
@pytest.mark.parametrize("name", sorted(BOX))
def test_flux_ranges(cuda, name, ratio):
    import torch
    cfg = BOX[name]
    rng = np.random.default_rng(int(1000 * ratio))
    K = (cfg["order"] + 1) ** cfg["dim"]
    shape = (int(np.prod(cfg["nelem"])), K)
    ends = lambda: np.where(rng.random(shape) < 0.5, 1.0, ratio) * ratio ** (0.02 * rng.uniform(-1, 1, shape))
    rho, p = ends(), 3.0 * ends()
    vel = [0.5 + 0.3 * rng.uniform(-1, 1, shape) for _ in range(cfg["dim"])]
    u = cases.prim_to_cons(rho, vel, p, 1.4)
    op, orc = DGSEMOperator(**cfg), O.Oracle(threads=8, **cfg)
    du = torch.tensor(u.reshape(-1), dtype=torch.float64, device=cuda)
    out = torch.empty_like(du)
    op.Mult(du, out)
    torch.cuda.synchronize()
    ref = orc.Mult(u)
    r = np.abs(out.cpu().numpy() - ref).max() / np.abs(ref).max()
    print("flux ranges %s ratio %g: %.3e" % (name, ratio, r), flush=True)
    assert r <= 1e-12
