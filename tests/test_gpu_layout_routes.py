"""Which lane layout lanes = 0 stands for in binary32: requests for the queue stay on one lane
per trajectory, one launch takes the matrix-core layout; the same bits either way."""
import pytest

from helpers import bits_equal, problem
from simplediffeq_hip import _abi, runtime

pytestmark = pytest.mark.gpu

FIELDS = ("u_end", "t_end", "retcode", "naccept", "nreject")


def _glv(n, **kw):
    u0, r, A = problem(_abi.RHS_GLV16, n, seed=4)
    d = runtime.make_desc(_abi.ALG_ATSIT5, dtype=_abi.F32, rhs=_abi.RHS_GLV16, n_traj=n,
                          tspan=(0.0, 3.0), dt=0.1, abstol=1e-6, reltol=1e-6, **kw)
    return d, runtime.EnsembleBuffers(d, 16, u0, r, A, backend="torch", device="cuda:0")


@pytest.mark.parametrize("kw,lanes", [
    (dict(), 4), (dict(schedule=_abi.SCHED_ONE_LAUNCH), 4),
    (dict(schedule=_abi.SCHED_ONE_LAUNCH, chunk=16), 4),
    (dict(schedule=_abi.SCHED_PERSISTENT), 1), (dict(schedule=_abi.SCHED_STAGED), 1),
    (dict(grid=4), 1), (dict(chunk=16), 1), (dict(refill=8), 1)])
def test_requests_for_the_queue_stay_on_one_lane(ctx, kw, lanes):
    d, b = _glv(200, **kw)
    ctx.solve(d, b)
    assert ctx.stats()["lanes"] == lanes
    d, ref = _glv(200, schedule=_abi.SCHED_ONE_LAUNCH, lanes=1)
    ctx.solve(d, ref)
    for f in FIELDS:
        assert bits_equal(b.numpy(f), ref.numpy(f)), f
