"""The launch shape of a solve that names none follows its size (one launch while the
ensemble is a few times what fits the GPU at once, then staged or persistent); whatever it
picks, the results are those of the persistent schedule, bit for bit, on every path: device
and host memory, the allocation-free solve, a replayed graph, a planned order."""
import numpy as np
import pytest

from helpers import bits_equal
from simplediffeq_hip import _abi, inputs, runtime

pytestmark = pytest.mark.gpu

FIELDS = ("u_end", "t_end", "retcode", "naccept", "nreject")


def _same(a, b):
    for f in FIELDS:
        assert bits_equal(a.numpy(f), b.numpy(f)), f


def _desc(n, sched, alg=_abi.ALG_ATSIT5, **kw):
    return runtime.make_desc(alg, n_traj=n, tspan=(0.0, 0.6), dt=0.1, abstol=1e-7, reltol=1e-6,
                             schedule=sched, **kw)


def _dev(d, u0, p, ts=None, **kw):
    return runtime.EnsembleBuffers(d, 3, u0, p, tspan=ts, backend="torch", device="cuda:0", **kw)


def _resident(c):
    """Lanes of the binary64 ATsit5 kernel that fit the GPU at once."""
    u0, p = inputs.lorenz_wide(64)
    d = _desc(64, _abi.SCHED_PERSISTENT, block=256)
    c.solve(d, _dev(d, u0, p))
    return c.stats()["grid"] * 256


@pytest.mark.parametrize("spans", [False, True])
@pytest.mark.parametrize("times,add", [(0, 1), (0, 65), (1, 0), (1, 1), (3, 0), (3, 1)])
def test_default_equals_persistent(times, add, spans):
    c = runtime.Context(0)  # nothing tuned
    n = times * _resident(c) + add
    u0, p = inputs.lorenz_wide(n, seed=6)
    ts = None
    if spans:
        ts = np.zeros((2, n))
        ts[1] = np.linspace(0.0, 0.6, n)
    ref = _dev(_desc(n, _abi.SCHED_PERSISTENT), u0, p, ts)
    c.solve(ref.desc, ref)
    got = _dev(_desc(n, _abi.SCHED_AUTO), u0, p, ts)
    c.solve(got.desc, got)
    _same(got, ref)
    want = _abi.SCHED_ONE_LAUNCH
    if spans and (times, add) == (3, 1):
        want = _abi.SCHED_PERSISTENT
    if not spans and (times, add) > (1, 0):
        want = _abi.SCHED_STAGED
    assert c.stats()["schedule"] == want
    assert c.stats()["block"] == (64 if want == _abi.SCHED_ONE_LAUNCH else 256)
    static = _dev(_desc(n, _abi.SCHED_AUTO), u0, p, ts)
    c.solve_static(static.desc, static)
    _same(static, ref)
    replay = _dev(_desc(n, _abi.SCHED_AUTO), u0, p, ts)
    h = c.graph_capture(replay.desc, replay)
    for _ in range(3):
        replay.u_end.zero_()
        c.graph_launch(h)
        c.synchronize()
        _same(replay, ref)
    c.graph_destroy(h)
    host = runtime.EnsembleBuffers(_desc(n, _abi.SCHED_AUTO), 3, u0, p, tspan=ts)
    c.solve(host.desc, host)
    _same(host, ref)
    c.close()


@pytest.mark.parametrize("dtype", [_abi.F64, _abi.F32])
@pytest.mark.parametrize("n", [65, 300_001])
def test_planned_order_default_equals_persistent(n, dtype):
    import torch
    c = runtime.Context(0)
    u0, p = inputs.lorenz_wide(n, seed=7)
    key = torch.as_tensor(np.random.default_rng(3).normal(-3.0, 1.0, n).astype(np.float32),
                          device="cuda:0")
    order = torch.empty(n, dtype=torch.int64, device="cuda:0")
    ref = _dev(_desc(n, _abi.SCHED_PERSISTENT, dtype=dtype), u0, p)
    c.solve(ref.desc, ref)
    got = _dev(_desc(n, _abi.SCHED_AUTO, dtype=dtype), u0, p, order=order)
    torch.cuda.synchronize()
    c.plan_order(key.data_ptr(), n, order.data_ptr())
    c.solve(got.desc, got)
    assert c.stats()["schedule"] == _abi.SCHED_ONE_LAUNCH
    _same(got, ref)
    c.close()


@pytest.mark.parametrize("lanes", [4, 16])
def test_persistent_default_chunk_of_group_layouts(lanes):
    """Beyond four times what fits, the layouts with several lanes per trajectory claim one
    wave's slots at a time."""
    c = runtime.Context(0)
    u0, r, A = inputs.glv16(64, seed=1)
    kw = dict(rhs=_abi.RHS_GLV16, tspan=(0.0, 0.2), dt=0.1, abstol=1e-6, reltol=1e-6, lanes=lanes)
    d = runtime.make_desc(_abi.ALG_ATSIT5, n_traj=64, schedule=_abi.SCHED_PERSISTENT, **kw)
    b = runtime.EnsembleBuffers(d, 16, u0, r, A, backend="torch", device="cuda:0")
    c.solve(d, b)
    n = 4 * c.stats()["grid"] * 256 // lanes + 1
    u0, r = np.resize(u0, (16, n)), np.resize(r, (16, n))
    out = []
    for sched in (_abi.SCHED_ONE_LAUNCH, _abi.SCHED_AUTO):
        d = runtime.make_desc(_abi.ALG_ATSIT5, n_traj=n, schedule=sched, **kw)
        b = runtime.EnsembleBuffers(d, 16, u0, r, A, backend="torch", device="cuda:0")
        c.solve(d, b)
        out.append(b)
    st = c.stats()
    assert st["schedule"] == _abi.SCHED_PERSISTENT and st["chunk"] == 64 // lanes
    _same(out[1], out[0])
    c.close()


def test_visit_counters_and_queue_fields_keep_the_queue(ctx):
    """A caller's own queue grid, chunk or refill batch is used; with visit counters each
    trajectory is taken up once, also where the default would be staged."""
    import torch
    n = _resident(ctx) + 1
    u0, p = inputs.lorenz_wide(n, seed=8)
    for kw in (dict(grid=40), dict(chunk=16), dict(refill=8)):
        d = _desc(2000, _abi.SCHED_AUTO, alg=_abi.ALG_AVERN9, **kw)
        c = runtime.Context(0)
        c.solve(d, _dev(d, u0[:, :2000], p[:, :2000]))
        assert c.stats()["schedule"] == _abi.SCHED_PERSISTENT
        for f, v in kw.items():
            assert c.stats()[f] == v
        c.close()
    c = runtime.Context(0)
    d = _desc(n, _abi.SCHED_AUTO)
    b = _dev(d, u0, p)
    seen = torch.zeros(n, dtype=torch.int32, device="cuda:0")
    b.io.visits = seen.data_ptr()
    torch.cuda.synchronize()
    c.solve(d, b)
    assert (seen.cpu().numpy() == 1).all()
    c.close()


@pytest.mark.parametrize("lanes,sched,more,chunk", [
    (4, _abi.SCHED_PERSISTENT, {}, 16), (16, _abi.SCHED_PERSISTENT, {}, 4),
    (4, _abi.SCHED_AUTO, dict(refill=2), 16), (16, _abi.SCHED_STAGED, {}, 4),
    (4, _abi.SCHED_PERSISTENT, dict(chunk=64), 64), (1, _abi.SCHED_PERSISTENT, {}, 64)])
def test_a_wave_claims_its_slots_where_the_queue_is_asked_for(ctx, lanes, sched, more, chunk):
    """A wave that claimed several waves' slots at a time left others without work."""
    n = 4001
    u0, r, A = inputs.glv16(n, seed=1)
    out = []
    for s, kw in ((_abi.SCHED_ONE_LAUNCH, {}), (sched, more)):
        d = runtime.make_desc(_abi.ALG_ATSIT5, rhs=_abi.RHS_GLV16, n_traj=n, tspan=(0.0, 2.0),
                              dt=0.1, abstol=1e-6, reltol=1e-6, lanes=lanes, schedule=s, **kw)
        b = runtime.EnsembleBuffers(d, 16, u0, r, A, backend="torch", device="cuda:0")
        ctx.solve(d, b)
        out.append(b)
    assert ctx.stats()["schedule"] == _abi.SCHED_PERSISTENT and ctx.stats()["chunk"] == chunk
    _same(out[1], out[0])
