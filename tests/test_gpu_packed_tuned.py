"""Packed save_everystep in a tuned context: tuning fixed rows, or a packed solve too small for
the ranked passes, leaves a large packed solve on its default passes, and a tuned large one
runs what the tuner found best.  Every way the same rows."""
import numpy as np
import pytest

from helpers import bits_equal
from simplediffeq_hip import _abi, runtime

pytestmark = pytest.mark.gpu

N = 400_001  # beyond what fits the GPU at once
SHAPE = ("schedule", "block", "grid", "chunk", "refill", "waves", "per_lane", "lanes")


def _inputs(n):
    """Few long trajectories among short ones, in no order: the queue beats one launch."""
    rng = np.random.default_rng(1)
    u0 = rng.uniform(-1.0, 1.0, (3, n))
    p = np.stack([rng.uniform(8.0, 12.0, n), rng.uniform(0.0, 20.0, n), rng.uniform(2.0, 3.0, n)])
    ts = np.zeros((2, n))
    ts[1] = np.where(rng.uniform(size=n) < 0.05, 3.0, 0.1)
    return u0, p, ts


def _bufs(n, packed, cap=0):
    u0, p, ts = _inputs(n)
    d = runtime.make_desc(_abi.ALG_ATSIT5, n_traj=n, dt=0.1, abstol=1e-6, reltol=1e-5,
                          span_order=1, save_everystep=True, max_saves=0 if packed else 150,
                          save_layout=_abi.SAVE_PACKED if packed else _abi.SAVE_TRAJ_MAJOR)
    return d, runtime.EnsembleBuffers(d, 3, u0, p, tspan=ts, backend="torch", device="cuda:0",
                                      steps_capacity=cap)


@pytest.fixture(scope="module")
def untuned():
    c = runtime.Context(0)
    d, b = _bufs(N, True)
    c.solve(d, b, allow=(_abi.E_SAVE_OVERFLOW,))
    d, b = _bufs(N, True, int(c.stats()["steps_needed"]))
    c.solve(d, b)
    st = c.stats()
    assert st["schedule"] == _abi.SCHED_ONE_LAUNCH and st["block"] == 256
    c.close()
    return b, st


def _same(a, b):
    for f in ("u_end", "t_end", "retcode", "naccept", "nreject", "n_steps", "steps_offset",
              "u_steps", "t_steps"):
        assert bits_equal(a.numpy(f), b.numpy(f)), f


@pytest.mark.parametrize("n,packed", [(60_001, False), (N, False), (1000, True)])
def test_other_tunings_leave_the_default_passes(untuned, n, packed):
    ref, st0 = untuned
    c = runtime.Context(0)
    d, b = _bufs(n, packed, 150 * n if packed else 0)
    best = c.autotune(d, b)
    if n == N:
        assert best["schedule"] == _abi.SCHED_PERSISTENT
    del b
    d, b = _bufs(N, True, ref.steps_capacity)
    c.solve(d, b)
    st = c.stats()
    assert [st[k] for k in SHAPE if k != "chunk"] == [st0[k] for k in SHAPE if k != "chunk"]
    _same(b, ref)
    c.close()


def test_a_tuned_packed_solve_runs_the_winner(untuned):
    ref, _ = untuned
    c = runtime.Context(0)
    d, b = _bufs(N, True, ref.steps_capacity)
    best = c.autotune(d, b)
    c.solve(d, b)
    st = c.stats()
    assert [st[k] for k in SHAPE if k != "chunk"] == [best[k] for k in SHAPE if k != "chunk"]
    _same(b, ref)
    c.close()
