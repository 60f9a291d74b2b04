"""Ensembles on both sides of the size at which their tiles change from node
threads to line threads, bit for bit against each case stepped alone."""
import pytest

from test_gpu_ensemble import assert_same, run_pair, step_sizes

pytestmark = pytest.mark.gpu

# elements a side of two cases: below and above
SIDES = {2: (56, 60), 3: (45, 48), 4: (39, 43), 5: (34, 37)}


@pytest.mark.parametrize("mode", [None, 2])
@pytest.mark.parametrize("blending", [False, True])
@pytest.mark.parametrize("order,n", [(N, n) for N in SIDES for n in SIDES[N]])
def test_sizes(cuda, order, n, blending, mode):
    cl = [dict(dim=2, order=order, nelem=(n, n), lo=(-1.0, -1.0), hi=(1.0, 1.0), gamma=1.4, precision="mixed", kind="kh",
               param=12.0 + i, seed=5 + i, blending=blending, alpha_max=0.5) for i in range(2)]
    d = step_sizes(cl)
    ue, us, ok = run_pair(cl, cuda, [d, d], mode=mode)
    assert_same(ue, us, cl)
    assert all(ok)
