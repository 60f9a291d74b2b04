"""The device time loop around its chunks of 8 steps and its graph (64 steps
to go): max_steps below, at and above them, and an end time that falls inside a
chunk, on a stream and on the default one, bitwise equal to single steps."""
import pytest

from prandtl_amd import DGSEMOperator, cases

pytestmark = pytest.mark.gpu

CFG = dict(dim=2, order=2, nelem=(6, 5), lo=(-5.0, -5.0), hi=(5.0, 5.0), quirks=False)
DT = 2.0 ** -9


@pytest.mark.parametrize("stream", [False, True])
@pytest.mark.parametrize("steps,by_time", [(1, False), (8, False), (9, False), (17, False), (90, False), (3, True), (8, True),
                                           (21, True), (150, True)])
def test_loop_chunks(cuda, steps, by_time, stream):
    import torch
    X = cases.node_coords(2, 2, CFG["nelem"], CFG["lo"], CFG["hi"])
    u0 = torch.tensor(cases.isentropic_vortex(X).reshape(-1), dtype=torch.float64, device=cuda)
    torch.cuda.synchronize()
    with torch.cuda.stream(torch.cuda.Stream() if stream else torch.cuda.default_stream()):
        a, b = u0.clone(), u0.clone()
        op, ref = DGSEMOperator(**CFG), DGSEMOperator(**CFG)
        t, n = op.Run(a, 0.0, steps * DT if by_time else 1e9, dt=DT, max_steps=0 if by_time else steps)
        for _ in range(steps):
            ref.Step(b, DT)
        torch.cuda.synchronize()
    assert n == steps and t == steps * DT
    assert torch.equal(a, b)
