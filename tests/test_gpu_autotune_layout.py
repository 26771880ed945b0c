"""The autotuner times one layout: the one that the solve taking its result runs on, also where
lanes = 0 stands for different layouts under different schedules (binary32 GLV-16)."""
import pytest

from helpers import problem
from simplediffeq_hip import _abi, runtime

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,lanes", [(_abi.F32, 4), (_abi.F64, 4)])
def test_every_candidate_runs_on_the_tuned_layout(dtype, lanes):
    import torch
    c = runtime.Context(0)
    n = 300
    u0, r, A = problem(_abi.RHS_GLV16, n, seed=4)
    d = runtime.make_desc(_abi.ALG_ATSIT5, dtype=dtype, rhs=_abi.RHS_GLV16, n_traj=n,
                          tspan=(0.0, 1.0), dt=0.1, abstol=1e-6, reltol=1e-6)
    b = runtime.EnsembleBuffers(d, 16, u0, r, A, backend="torch", device="cuda:0")
    seen = torch.zeros(n, dtype=torch.int32, device="cuda:0")
    b.io.visits = seen.data_ptr()
    torch.cuda.synchronize()
    best = c.autotune(d, b)
    # three one-launch and ten persistent shapes, twice each: nothing that needs one lane
    assert (seen.cpu().numpy() == 26).all()
    assert best["lanes"] == lanes
    c.solve(d, b)
    st = c.stats()
    for f in ("schedule", "lanes", "block", "chunk", "waves", "per_lane", "refill"):
        assert st[f] == best[f], f
    c.close()
