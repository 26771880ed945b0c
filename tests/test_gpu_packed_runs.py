"""Packed save_everystep rows: states on both sides of the 32-byte rule, sizes around a wave
and a block, both precisions, a trajectory left with part of its rows (against the
trajectory-major rows, bit for bit); and, beyond what fits the GPU at once, the saving pass
in the order of the counted attempts that writes whole sectors from LDS
(against the persistent schedule, bit for bit)."""
import numpy as np
import pytest

from helpers import bits_equal, problem
from simplediffeq_hip import _abi, runtime, tracer

pytestmark = pytest.mark.gpu


def _rhs(ctx, n_state):
    """A right-hand side of n_state components (built in where there is one)."""
    builtin = {1: (_abi.RHS_AFFINE1, 2), 2: (_abi.RHS_LINEAR2, 4), 3: (_abi.RHS_LORENZ, 3)}
    if n_state in builtin:
        return builtin[n_state]

    def f(u, p, t):
        return [p[0] * (u[(i + 1) % n_state] - u[i]) for i in range(n_state)]
    src, fn = tracer.trace(f, n_state, 1, "packed_runs_%d" % n_state)
    return ctx.compile_rhs(src, fn, n_state, 1), 1


def _pair(c, n, n_state, rhs, n_param, alg, dtype, cap=None, sched=_abi.SCHED_AUTO):
    rng = np.random.default_rng(n + n_state)
    u0 = rng.uniform(-1.0, 1.0, (n_state, n))
    p = rng.uniform(0.5, 3.0, (n_param, n))
    kw = dict(rhs=rhs, n_traj=n, tspan=(0.0, 1.0), abstol=1e-8, reltol=1e-7, dtype=dtype,
                   dt=0.1 if alg in _abi.ADAPTIVE_ALGS else 0.0625, save_everystep=True)
    d = runtime.make_desc(alg, save_layout=_abi.SAVE_TRAJ_MAJOR, max_saves=400,
                          schedule=_abi.SCHED_ONE_LAUNCH, **kw)
    ref = runtime.EnsembleBuffers(d, n_state, u0, p)
    c.solve(d, ref)
    rows = int(ref.n_steps.sum())
    d = runtime.make_desc(alg, save_layout=_abi.SAVE_PACKED, schedule=sched, **kw)
    g = runtime.EnsembleBuffers(d, n_state, u0, p, steps_capacity=rows if cap is None else cap(rows))
    g.u_steps[:] = -5.5
    g.t_steps[:] = -5.5
    st = c.solve(d, g, allow=(_abi.E_SAVE_OVERFLOW,))
    assert st == (0 if cap is None else _abi.E_SAVE_OVERFLOW)
    return ref, g


def _same_rows(ref, g, n):
    off, k = g.steps_offset, g.n_steps
    assert off[0] == 0 and np.array_equal(np.diff(off), k)
    keep = np.arange(ref.t_steps.shape[1])[None, :] < k[:, None]
    used = int(off[n])
    assert bits_equal(g.t_steps[:used], ref.t_steps[keep])
    assert bits_equal(g.u_steps[:used], ref.u_steps[keep])
    assert (g.t_steps[used:] == -5.5).all() and (g.u_steps[used:] == -5.5).all()


@pytest.mark.parametrize("n", [1, 63, 65, 257, 1000])
@pytest.mark.parametrize("alg", [_abi.ALG_ATSIT5, _abi.ALG_AVERN7, _abi.ALG_TSIT5, _abi.ALG_RK4])
@pytest.mark.parametrize("n_state,dtype", [(1, _abi.F64), (2, _abi.F64), (3, _abi.F64),
                                           (3, _abi.F32), (1, _abi.F32)])
def test_runs_equal_trajectory_major_rows(ctx, n_state, dtype, alg, n):
    rhs, n_param = _rhs(ctx, n_state)
    ref, g = _pair(ctx, n, n_state, rhs, n_param, alg, dtype)
    assert np.array_equal(g.n_steps, ref.n_steps)
    _same_rows(ref, g, n)


@pytest.mark.parametrize("n_state,dtype", [(4, _abi.F64), (5, _abi.F64), (8, _abi.F32), (9, _abi.F32)])
@pytest.mark.parametrize("sched", [_abi.SCHED_AUTO, _abi.SCHED_PERSISTENT])
def test_runs_of_traced_states(ctx, n_state, dtype, sched):
    rhs, n_param = _rhs(ctx, n_state)
    ref, g = _pair(ctx, 300, n_state, rhs, n_param, _abi.ALG_ATSIT5, dtype, sched=sched)
    _same_rows(ref, g, 300)


@pytest.mark.parametrize("alg", [_abi.ALG_ATSIT5, _abi.ALG_TSIT5])
@pytest.mark.parametrize("short", [1, 2, 3, 1001])
def test_cut_in_the_middle_of_a_run(ctx, alg, short):
    ref, g = _pair(ctx, 200, 3, _abi.RHS_LORENZ, 3, alg, _abi.F64, cap=lambda r: r - short)
    _same_rows(ref, g, 200)


@pytest.mark.parametrize("n_state,dtype,alg,spans,cut", [
    (3, _abi.F64, _abi.ALG_ATSIT5, False, 0), (3, _abi.F64, _abi.ALG_ATSIT5, True, 1001),
    (3, _abi.F32, _abi.ALG_ATSIT5, False, 1001), (3, _abi.F32, _abi.ALG_AVERN7, True, 0),
    (1, _abi.F64, _abi.ALG_AVERN7, True, 0), (2, _abi.F64, _abi.ALG_AVERN9, False, 2),
    (4, _abi.F64, _abi.ALG_ATSIT5, True, 3)])
def test_ranked_saving_pass(n_state, dtype, alg, spans, cut):
    """Beyond what fits the GPU at once the saving pass takes the trajectories by their
    counted attempts and writes sector by sector; everything is the persistent schedule's."""
    c = runtime.Context(0)
    rhs, n_param = _rhs(c, n_state)
    n = 600_001
    rng = np.random.default_rng(n_state)
    u0 = rng.uniform(-1.0, 1.0, (n_state, n))
    p = rng.uniform(0.5, 3.0, (n_param, n))
    ts = None
    if spans:
        ts = np.zeros((2, n))
        ts[1] = rng.permutation(np.linspace(0.0, 0.8, n))
    out, rows = [], n * 30
    for sched in (_abi.SCHED_PERSISTENT, _abi.SCHED_PERSISTENT, _abi.SCHED_AUTO):
        d = runtime.make_desc(alg, rhs=rhs, n_traj=n, tspan=(0.0, 0.8), dt=0.1, abstol=1e-6,
                              reltol=1e-4, dtype=dtype, schedule=sched, save_everystep=True,
                              save_layout=_abi.SAVE_PACKED)
        b = runtime.EnsembleBuffers(d, n_state, u0, p, tspan=ts, backend="torch",
                                    device="cuda:0", steps_capacity=rows)
        b.u_steps.fill_(-5.5)
        b.t_steps.fill_(-5.5)
        st = c.solve(d, b, allow=(_abi.E_SAVE_OVERFLOW,))
        assert st == (_abi.E_SAVE_OVERFLOW if cut and len(out) else 0)
        rows = int(c.stats()["steps_needed"]) - cut
        out.append(b)
    assert c.stats()["schedule"] == _abi.SCHED_ONE_LAUNCH
    for f in ("u_end", "t_end", "retcode", "naccept", "nreject", "n_steps", "steps_offset",
              "u_steps", "t_steps"):
        assert bits_equal(out[1].numpy(f), out[2].numpy(f)), f
    c.close()
