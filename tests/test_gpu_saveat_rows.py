"""Point-major saveat output beyond 300 MiB: by way of trajectory-major rows and a transpose,
the trajectory-major solve's values bit for bit, at sizes off the transpose's tiles, with
trajectories that end early, in both precisions; and a planned order that leaves trajectories
out leaves their rows NaN."""
import numpy as np
import pytest

from helpers import problem
from simplediffeq_hip import _abi, runtime

pytestmark = pytest.mark.gpu


def _solve(c, rhs, alg, dtype, n, points, layout, u0, p, ps, ts, order=None):
    import torch
    d = runtime.make_desc(alg, dtype=dtype, rhs=rhs, n_traj=n, tspan=(0.0, 2.0), dt=0.1,
                          abstol=1e-6, reltol=1e-4, saveat=np.linspace(0.0, 2.0, points),
                          save_layout=layout)
    b = runtime.EnsembleBuffers(d, u0.shape[0], u0, p, ps, ts, order=order, backend="torch",
                                device="cuda:0")
    b.u_saveat.fill_(-77.25)
    torch.cuda.synchronize()
    assert c.solve(d, b) == 0
    return b


@pytest.mark.parametrize("rhs,alg,dtype,n,points", [
    (_abi.RHS_LORENZ, _abi.ALG_ATSIT5, _abi.F64, 130_003, 101),
    (_abi.RHS_LORENZ, _abi.ALG_ATSIT5, _abi.F32, 327_745, 81),
    (_abi.RHS_LORENZ, _abi.ALG_AVERN7, _abi.F64, 81_921, 161),
    (_abi.RHS_GLV16, _abi.ALG_ATSIT5, _abi.F32, 40_127, 128),
    (_abi.RHS_GLV16, _abi.ALG_ATSIT5, _abi.F64, 25_601, 97)])
def test_rows_are_the_trajectory_major_solve(rhs, alg, dtype, n, points):
    import torch
    c = runtime.Context(0)
    u0, p, ps = problem(rhs, n, seed=points)
    ts = np.zeros((2, n))
    ts[1] = np.linspace(0.0, 2.2, n)
    a = _solve(c, rhs, alg, dtype, n, points, _abi.SAVE_POINT_MAJOR, u0, p, ps, ts)
    b = _solve(c, rhs, alg, dtype, n, points, _abi.SAVE_TRAJ_MAJOR, u0, p, ps, ts)
    assert a.u_saveat.numel() * a.u_saveat.element_size() > 300 << 20
    it = torch.int64 if dtype == _abi.F64 else torch.int32
    assert torch.equal(a.u_saveat.view(it), b.u_saveat.permute(1, 2, 0).contiguous().view(it))
    assert torch.isnan(a.u_saveat).any()
    for f in ("u_end", "t_end", "naccept"):
        assert torch.equal(getattr(a, f), getattr(b, f)), f
    c.close()


def test_rows_of_trajectories_left_out_are_nan():
    import torch
    c = runtime.Context(0)
    n, points = 131_072, 101
    u0, p, ps = problem(_abi.RHS_LORENZ, n, seed=9)
    dev = torch.device("cuda:0")
    key = torch.as_tensor(-np.random.default_rng(2).normal(3.0, 1.0, n).astype(np.float32),
                          device=dev)
    order = torch.empty(n, dtype=torch.int64, device=dev)
    torch.cuda.synchronize()
    c.plan_order(key.data_ptr(), n, order.data_ptr())
    c.synchronize()
    lost, kept = int(order[5]), int(order[7])
    order[5] = order[7]
    torch.cuda.synchronize()
    b = _solve(c, _abi.RHS_LORENZ, _abi.ALG_ATSIT5, _abi.F64, n, points, _abi.SAVE_POINT_MAJOR,
               u0, p, ps, None, order=order)
    assert torch.isnan(b.u_saveat[:, :, lost]).all()
    assert torch.isfinite(b.u_saveat[:, :, kept]).all()
    c.close()


# Which solves take the rows: told by the context's scratch, which holds them.  Half of the
# save times have to lie in the span, and in an order, where no store shares a line with
# another lane's, fewer save times do.  Either way the trajectory-major solve's values.
@pytest.mark.parametrize("alg,dtype,n,points,last,order,rows", [
    (_abi.ALG_ATSIT5, _abi.F64, 130_003, 101, 2.0, False, True),
    (_abi.ALG_AVERN7, _abi.F64, 81_921, 161, 2.0, False, True),
    (_abi.ALG_ATSIT5, _abi.F64, 90_001, 161, 4.0, False, True),    # 81 reached
    (_abi.ALG_ATSIT5, _abi.F64, 90_001, 161, 4.1, False, False),   # 79 reached
    (_abi.ALG_ATSIT5, _abi.F64, 60_001, 400, 8.0, False, False),   # 100 of 400
    (_abi.ALG_ATSIT5, _abi.F32, 781_253, 32, 2.0, True, True),
    (_abi.ALG_ATSIT5, _abi.F32, 806_455, 31, 2.0, True, False),
    (_abi.ALG_AVERN7, _abi.F32, 247_524, 101, 2.0, True, False),    # just below the line
    (_abi.ALG_AVERN7, _abi.F32, 247_525, 101, 2.0, True, True),     # just above
    (_abi.ALG_ATSIT5, _abi.F64, 130_003, 101, 2.0, True, False)])
def test_which_solves_take_the_rows(alg, dtype, n, points, last, order, rows):
    import torch
    u0, p, ps = problem(_abi.RHS_LORENZ, n, seed=points)
    o = np.random.default_rng(3).permutation(n) if order else None
    out, used = [], 0
    for layout in (_abi.SAVE_POINT_MAJOR, _abi.SAVE_TRAJ_MAJOR):
        d = runtime.make_desc(alg, dtype=dtype, n_traj=n, tspan=(0.0, 2.0), dt=0.1, abstol=1e-6,
                              reltol=1e-4, saveat=np.linspace(0.0, last, points),
                              save_layout=layout)
        b = runtime.EnsembleBuffers(d, 3, u0, p, order=o, backend="torch", device="cuda:0")
        b.u_saveat.fill_(-77.25)
        c = runtime.Context(0)
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        assert c.solve(d, b) == 0
        if layout == _abi.SAVE_POINT_MAJOR:
            used = before - torch.cuda.mem_get_info()[0]
        c.close()
        out.append(b.u_saveat.view(torch.int64 if dtype == _abi.F64 else torch.int32))
    assert torch.equal(out[0], out[1].permute(1, 2, 0).contiguous())
    assert (used >= out[0].numel() * out[0].element_size()) == rows


def test_rows_of_trajectories_left_out_of_an_order_are_nan():
    import torch
    c = runtime.Context(0)
    n, points = 262_147, 101
    u0, p, ps = problem(_abi.RHS_LORENZ, n, seed=10)
    dev = torch.device("cuda:0")
    key = torch.as_tensor(-np.random.default_rng(4).normal(3.0, 1.0, n).astype(np.float32),
                          device=dev)
    order = torch.empty(n, dtype=torch.int64, device=dev)
    torch.cuda.synchronize()
    c.plan_order(key.data_ptr(), n, order.data_ptr())
    c.synchronize()
    lost, kept = int(order[5]), int(order[7])
    order[5] = order[7]
    torch.cuda.synchronize()
    b = _solve(c, _abi.RHS_LORENZ, _abi.ALG_ATSIT5, _abi.F64, n, points, _abi.SAVE_POINT_MAJOR,
               u0, p, ps, None, order=order)
    assert torch.isnan(b.u_saveat[:, :, lost]).all()
    assert torch.isfinite(b.u_saveat[:, :, kept]).all()
    c.close()
