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
