"""Saveat rows that a trajectory does not reach are NaN whatever the output buffer held
before: trajectories that end before the last save time (their own t_end, the attempt
limit, an empty span), in every lane layout, both save layouts and the fixed-step
solvers, bit for bit against the CPU oracle; and trajectories that an overwritten planned
order leaves out."""
import numpy as np
import pytest

from helpers import assert_bit_identical, problem
from simplediffeq_hip import _abi, runtime

pytestmark = pytest.mark.gpu

POISON = -77.25


def _solve_pair(ctx, d, n_state, u0, p, ps=None, ts=None):
    import torch
    from oracle import pyoracle
    g = runtime.EnsembleBuffers(d, n_state, u0, p, ps, ts, backend="torch", device="cuda:0")
    g.u_saveat.fill_(POISON)
    torch.cuda.synchronize()
    ctx.solve(d, g)
    c = runtime.EnsembleBuffers(d, n_state, u0, p, ps, ts)
    pyoracle.solve(d, c, nthreads=8)
    return g, c


@pytest.mark.parametrize("layout", [_abi.SAVE_POINT_MAJOR, _abi.SAVE_TRAJ_MAJOR])
@pytest.mark.parametrize("rhs,alg,lanes", [(_abi.RHS_LORENZ, _abi.ALG_ATSIT5, 1),
                                           (_abi.RHS_LORENZ, _abi.ALG_AVERN7, 1),
                                           (_abi.RHS_GLV16, _abi.ALG_AVERN9, 4),
                                           (_abi.RHS_GLV16, _abi.ALG_ATSIT5, 16)])
def test_rows_after_the_end_are_nan(ctx, rhs, alg, lanes, layout):
    n, saveat = 203, np.linspace(0.0, 6.0, 37)
    u0, p, ps = problem(rhs, n, seed=7)
    ts = np.zeros((2, n))
    ts[1] = np.linspace(0.0, 6.5, n)  # from an empty span to past the last save time
    d = runtime.make_desc(alg, rhs=rhs, n_traj=n, dt=0.1, abstol=1e-7, reltol=1e-7, maxiters=25,
                          saveat=saveat, lanes=lanes, save_layout=layout)
    g, c = _solve_pair(ctx, d, u0.shape[0], u0, p, ps, ts)
    assert_bit_identical(g, c, ("u_end", "t_end", "retcode", "naccept", "u_saveat"))
    rows = g.numpy("u_saveat")
    assert np.isnan(rows).any() and not (rows == POISON).any()


@pytest.mark.parametrize("layout", [_abi.SAVE_POINT_MAJOR, _abi.SAVE_TRAJ_MAJOR])
@pytest.mark.parametrize("alg", [_abi.ALG_TSIT5, _abi.ALG_VERN7, _abi.ALG_VERN9])
def test_fixed_step_rows_past_the_grid_are_nan(ctx, alg, layout):
    n = 131
    u0, p, _ = problem(_abi.RHS_LORENZ, n, seed=8)
    d = runtime.make_desc(alg, n_traj=n, tspan=(0.0, 1.0), dt=0.05, save_layout=layout,
                          saveat=np.linspace(0.0, 2.0, 21))
    g, c = _solve_pair(ctx, d, 3, u0, p)
    assert_bit_identical(g, c, ("u_end", "u_saveat"))
    assert np.isnan(g.numpy("u_saveat")).any()


def test_rows_of_trajectories_left_out_are_nan(ctx):
    import torch
    n = 4096
    u0, p, _ = problem(_abi.RHS_LORENZ, n, seed=9)
    dev = torch.device("cuda:0")
    key = torch.as_tensor(-np.random.default_rng(2).normal(3.0, 1.0, n).astype(np.float32),
                          device=dev)
    order = torch.empty(n, dtype=torch.int64, device=dev)
    torch.cuda.synchronize()
    ctx.plan_order(key.data_ptr(), n, order.data_ptr())
    ctx.synchronize()
    lost = int(order[5])
    order[5] = n + 3
    d = runtime.make_desc(_abi.ALG_ATSIT5, n_traj=n, tspan=(0.0, 1.0), dt=0.1,
                          saveat=[0.25, 0.5, 1.0], save_layout=_abi.SAVE_TRAJ_MAJOR)
    b = runtime.EnsembleBuffers(d, 3, u0, p, order=order, backend="torch", device=dev)
    assert b.order.data_ptr() == order.data_ptr()
    b.u_saveat.fill_(POISON)
    torch.cuda.synchronize()
    ctx.solve(d, b)
    rows = b.numpy("u_saveat")
    assert np.isnan(rows[lost]).all()
    assert np.isfinite(np.delete(rows, lost, axis=0)).all()


# The save times' share beyond the end decides whether the rows not reached are written by
# the trajectories or beforehand: both sides of the line, and trajectories that end before
# their span does, which no share foretells.
@pytest.mark.parametrize("layout", [_abi.SAVE_POINT_MAJOR, _abi.SAVE_TRAJ_MAJOR])
@pytest.mark.parametrize("rhs,alg,dtype,lanes", [
    (_abi.RHS_LORENZ, _abi.ALG_ATSIT5, _abi.F64, 1),
    (_abi.RHS_LORENZ, _abi.ALG_AVERN9, _abi.F64, 1),
    (_abi.RHS_LORENZ, _abi.ALG_AVERN7, _abi.F32, 1),
    (_abi.RHS_GLV16, _abi.ALG_ATSIT5, _abi.F64, 4)])
@pytest.mark.parametrize("last,maxiters", [(1.0, 1000), (1.03, 1000), (1.1, 1000), (9.0, 1000),
                                           (1.0, 9), (9.0, 9)])
def test_rows_beyond_a_common_end_are_nan(ctx, rhs, alg, dtype, lanes, layout, last, maxiters):
    n, saveat = 331, np.linspace(0.0, last, 33)
    u0, p, ps = problem(rhs, n, seed=11)
    d = runtime.make_desc(alg, dtype=dtype, rhs=rhs, n_traj=n, tspan=(0.0, 1.0),
                          dt=float(np.float32(0.1)), abstol=1e-6, reltol=1e-5,
                          maxiters=maxiters, saveat=saveat,
                          lanes=lanes, save_layout=layout)
    g, c = _solve_pair(ctx, d, u0.shape[0], u0, p, ps)
    if dtype == _abi.F64:
        assert_bit_identical(g, c, ("u_end", "t_end", "retcode", "naccept", "u_saveat"))
    rows = g.numpy("u_saveat")
    rows = rows if layout == _abi.SAVE_TRAJ_MAJOR else np.moveaxis(rows, -1, 0)
    beyond = saveat[None, :] > g.numpy("t_end")[:, None]
    assert np.array_equal(np.isnan(rows), np.broadcast_to(beyond[:, :, None], rows.shape))
    assert not (rows == POISON).any()


@pytest.mark.parametrize("own", [False, True])
def test_rows_not_reached_are_nan_on_every_path(ctx, own):
    import torch
    n, saveat = 1003, np.linspace(0.0, 3.0, 17)
    u0, p, _ = problem(_abi.RHS_LORENZ, n, seed=12)
    ts = np.vstack([np.zeros(n), np.linspace(0.1, 3.2, n)]) if own else None
    d = runtime.make_desc(_abi.ALG_ATSIT5, n_traj=n, tspan=(0.0, 1.0), dt=0.1, abstol=1e-6,
                          reltol=1e-5, saveat=saveat)
    g, c = _solve_pair(ctx, d, 3, u0, p, None, ts)
    want = c.numpy("u_saveat")
    h = runtime.EnsembleBuffers(d, 3, u0, p, tspan=ts)
    h.u_saveat[...] = POISON
    ctx.solve(d, h)
    assert want.tobytes() == h.numpy("u_saveat").tobytes()
    for call in ("static", "graph"):
        g.u_saveat.fill_(POISON)
        torch.cuda.synchronize()
        if call == "static":
            ctx.solve_static(d, g)
        else:
            h = ctx.graph_capture(d, g)
            for _ in range(2):
                g.u_saveat.fill_(POISON)
                torch.cuda.synchronize()
                ctx.graph_launch(h)
                ctx.synchronize()
            ctx.graph_destroy(h)
        torch.cuda.synchronize()
        assert want.tobytes() == g.numpy("u_saveat").tobytes(), call
