"""Where the default launch shape leaves one launch for the queue: as soon as the ensemble does
not fit the GPU at once, unless the library orders it by its spans or the caller gives an order
(endpoint output), it runs several binary32 lanes per trajectory, or its output is dense.  On
ensembles whose trajectories differ in length one launch is slower there: saved output, unsorted
spans, the allocation-free solve, an order whose keys need not predict anything, the matrix-core
layout.  On both sides of each line the results are the explicit schedule's, bit for bit."""
import numpy as np
import pytest

from helpers import bits_equal
from simplediffeq_hip import _abi, inputs, runtime

pytestmark = pytest.mark.gpu

FIELDS = ("u_end", "t_end", "retcode", "naccept", "nreject")


def _inputs(rhs, n):
    if rhs == _abi.RHS_GLV16:
        u0, r, A = inputs.glv16(64, seed=1)
        return np.resize(u0, (16, n)), np.resize(r, (16, n)), A
    return inputs.lorenz_wide(n, seed=5) + (None,)


@pytest.mark.parametrize("add", [0, 1])
@pytest.mark.parametrize("name,rhs,alg,dtype,points,spans,times", [
    ("saveat", _abi.RHS_LORENZ, _abi.ALG_AVERN7, _abi.F64, 3, False, 1),
    ("saveat", _abi.RHS_LORENZ, _abi.ALG_ATSIT5, _abi.F32, 3, True, 1),
    ("static", _abi.RHS_LORENZ, _abi.ALG_ATSIT5, _abi.F64, 0, False, 1),
    ("static", _abi.RHS_LORENZ, _abi.ALG_AVERN7, _abi.F64, 0, True, 1),
    ("planned", _abi.RHS_LORENZ, _abi.ALG_ATSIT5, _abi.F64, 0, True, 1.5),
    ("planned", _abi.RHS_LORENZ, _abi.ALG_ATSIT5, _abi.F32, 0, True, 1.5),
    ("planned", _abi.RHS_LORENZ, _abi.ALG_ATSIT5, _abi.F32, 3, True, 1),
    ("lanes", _abi.RHS_GLV16, _abi.ALG_AVERN9, _abi.F64, 3, False, 1),
    ("lanes", _abi.RHS_GLV16, _abi.ALG_ATSIT5, _abi.F32, 0, False, 2)])
def test_one_launch_ends_where_unlike_lengths_lose(name, rhs, alg, dtype, points, spans, times,
                                                   add):
    import torch
    c = runtime.Context(0)
    kw = dict(rhs=rhs, dtype=dtype, tspan=(0.0, 0.3), dt=0.1, abstol=1e-6, reltol=1e-5,
              saveat=np.linspace(0.0, 0.3, points) if points else None)

    def solve(n, sched, order=None, **more):
        u0, p, ps = _inputs(rhs, n)
        ts = None
        if spans:
            ts = np.zeros((2, n))
            ts[1] = np.linspace(0.0, 0.3, n)
        d = runtime.make_desc(alg, n_traj=n, schedule=sched, **kw, **more)
        b = runtime.EnsembleBuffers(d, u0.shape[0], u0, p, ps, ts, order=order, backend="torch",
                                    device="cuda:0")
        torch.cuda.synchronize()
        if order is not None:
            key = torch.as_tensor(np.random.default_rng(3).normal(-3.0, 1.0, n).astype(np.float32),
                                  device="cuda:0")
            c.plan_order(key.data_ptr(), n, b.order.data_ptr())
        (c.solve_static if name == "static" else c.solve)(d, b)
        return b, c.stats()

    # the persistent grid is the lanes that fit the GPU at once
    lanes = 4 if rhs == _abi.RHS_GLV16 else 1
    _, st = solve(100, _abi.SCHED_PERSISTENT, lanes=lanes, block=256)
    n = int(times * st["grid"] * 256) // lanes + add
    order = torch.zeros(n, dtype=torch.int64, device="cuda:0") if name == "planned" else None
    got, st = solve(n, _abi.SCHED_AUTO, order)
    assert st["lanes"] == lanes
    assert st["schedule"] == (_abi.SCHED_PERSISTENT if add else _abi.SCHED_ONE_LAUNCH)
    ref, _ = solve(n, _abi.SCHED_ONE_LAUNCH if add else _abi.SCHED_PERSISTENT, lanes=lanes)
    for f in FIELDS + (("u_saveat",) if points else ()):
        assert bits_equal(got.numpy(f), ref.numpy(f)), f
    c.close()


@pytest.mark.parametrize("dtype,times,add,want", [
    (_abi.F64, 1, 0, _abi.SCHED_ONE_LAUNCH), (_abi.F64, 1, 1, _abi.SCHED_STAGED),
    (_abi.F64, 4, 0, _abi.SCHED_STAGED), (_abi.F64, 4, 1, _abi.SCHED_PERSISTENT),
    (_abi.F32, 1, 0, _abi.SCHED_ONE_LAUNCH), (_abi.F32, 1, 1, _abi.SCHED_PERSISTENT)])
def test_where_the_staged_schedule_is_taken(dtype, times, add, want):
    c = runtime.Context(0)

    def solve(n, sched, **more):
        u0, p = inputs.lorenz_wide(n, seed=5)
        d = runtime.make_desc(_abi.ALG_ATSIT5, n_traj=n, dtype=dtype, tspan=(0.0, 0.2), dt=0.1,
                              abstol=1e-6, reltol=1e-4, schedule=sched, **more)
        b = runtime.EnsembleBuffers(d, 3, u0, p, backend="torch", device="cuda:0")
        c.solve(d, b)
        return b, c.stats()

    _, st = solve(100, _abi.SCHED_PERSISTENT, block=256)
    n = times * st["grid"] * 256 + add
    got, st = solve(n, _abi.SCHED_AUTO)
    assert st["schedule"] == want
    ref, _ = solve(n, _abi.SCHED_ONE_LAUNCH)
    for f in FIELDS:
        assert bits_equal(got.numpy(f), ref.numpy(f)), f
    c.close()


@pytest.mark.parametrize("alg,kahan", [(_abi.ALG_ATSIT5, False), (_abi.ALG_AVERN7, False),
                                       (_abi.ALG_ATSIT5, True)])
@pytest.mark.parametrize("parked", ["none", "some", "all", "endless"])
@pytest.mark.parametrize("n", [2, 63, 65, 5003])
def test_a_staged_solve_resumes_exactly_the_parked(ctx, alg, kahan, parked, n):
    """Its second launch starts behind the trajectories that ended in the first: none, some or
    all of them, and trajectories whose estimate of the attempts still to come is infinite."""
    u0, p = inputs.lorenz_wide(n, seed=9)
    span = {"none": 0.01, "some": 3.0, "all": 30.0, "endless": 3.0}[parked]
    ts = np.zeros((2, n))
    ts[1] = np.linspace(0.0, span, n) if parked == "some" else span
    if parked == "endless":
        ts[1, ::3] = np.inf
    out = []
    for sched in (_abi.SCHED_ONE_LAUNCH, _abi.SCHED_STAGED):
        d = runtime.make_desc(alg, dtype=_abi.F32 if kahan else _abi.F64, n_traj=n, dt=0.1,
                              abstol=1e-7, reltol=1e-6, schedule=sched, maxiters=200,
                              precision=_abi.PREC_KAHAN if kahan else _abi.PREC_PLAIN)
        b = runtime.EnsembleBuffers(d, 3, u0, p, tspan=ts)
        ctx.solve(d, b, allow=(_abi.E_DTMIN,))
        assert ctx.stats()["schedule"] == sched
        out.append(b)
    att = out[0].naccept + out[0].nreject
    if parked == "none":
        assert att.max() < 32
    elif parked != "some":
        assert att.max() > 32
    for f in FIELDS:
        assert bits_equal(out[0].numpy(f), out[1].numpy(f)), f


@pytest.mark.parametrize("rhs,alg,points,layout,last,times,add,want", [
    (_abi.RHS_GLV16, _abi.ALG_AVERN9, 256, _abi.SAVE_POINT_MAJOR, 0.3, 1, 1, 1),
    (_abi.RHS_GLV16, _abi.ALG_AVERN9, 255, _abi.SAVE_POINT_MAJOR, 0.3, 1, 1, 2),
    (_abi.RHS_GLV16, _abi.ALG_AVERN9, 256, _abi.SAVE_TRAJ_MAJOR, 0.3, 1, 1, 2),
    (_abi.RHS_GLV16, _abi.ALG_AVERN9, 256, _abi.SAVE_POINT_MAJOR, 0.31, 1, 1, 2),
    (_abi.RHS_LORENZ, _abi.ALG_ATSIT5, 64, _abi.SAVE_POINT_MAJOR, 0.3, 4, 0, 1),
    (_abi.RHS_LORENZ, _abi.ALG_ATSIT5, 64, _abi.SAVE_POINT_MAJOR, 0.3, 4, 1, 2),
    (_abi.RHS_LORENZ, _abi.ALG_ATSIT5, 63, _abi.SAVE_POINT_MAJOR, 0.3, 2, 0, 2),
    (_abi.RHS_LORENZ, _abi.ALG_AVERN7, 150, _abi.SAVE_POINT_MAJOR, 0.3, 2, 0, 1)])
def test_dense_output_stored_in_place_keeps_one_launch(rhs, alg, points, layout, last, times,
                                                       add, want):
    import torch
    c = runtime.Context(0)

    def solve(n, sched, **more):
        u0, p, ps = _inputs(rhs, n)
        d = runtime.make_desc(alg, rhs=rhs, n_traj=n, tspan=(0.0, 0.3), dt=0.1, abstol=1e-6,
                              reltol=1e-5, saveat=np.linspace(0.0, last, points),
                              save_layout=layout, schedule=sched, **more)
        b = runtime.EnsembleBuffers(d, u0.shape[0], u0, p, ps, backend="torch", device="cuda:0")
        c.solve(d, b)
        return b, c.stats()

    lanes = 4 if rhs == _abi.RHS_GLV16 else 1
    _, st = solve(100, _abi.SCHED_PERSISTENT, lanes=lanes, block=256)
    n = times * st["grid"] * 256 // lanes + add
    got, st = solve(n, _abi.SCHED_AUTO)
    assert st["schedule"] == (_abi.SCHED_ONE_LAUNCH if want == 1 else _abi.SCHED_PERSISTENT)
    ref, _ = solve(n, _abi.SCHED_PERSISTENT if want == 1 else _abi.SCHED_ONE_LAUNCH, lanes=lanes)
    for f in FIELDS:
        assert bits_equal(got.numpy(f), ref.numpy(f)), f
    assert torch.equal(got.u_saveat.view(torch.int64), ref.u_saveat.view(torch.int64))
    c.close()
