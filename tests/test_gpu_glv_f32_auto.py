"""Binary32 GLV-16 with lanes = 0: beyond 64 trajectories ATsit5 takes the matrix-core layout,
with the bits of one lane per trajectory, at states and coefficients of every magnitude
(subnormal, overflowing, infinite, NaN), in both save layouts, and with trajectories that end
early; requests that only one lane per trajectory offers stay there."""
import numpy as np
import pytest

from helpers import bits_equal, problem
from simplediffeq_hip import _abi, runtime

pytestmark = pytest.mark.gpu

FIELDS = ("u_end", "t_end", "retcode", "naccept", "nreject")
ALLOW = (_abi.E_DTMIN,)


def _pair(ctx, u0, r, A, tspan=None, **kw):
    n = u0.shape[1]
    out, lanes = [], []
    for ln in (1, 0):
        d = runtime.make_desc(_abi.ALG_ATSIT5, dtype=_abi.F32, rhs=_abi.RHS_GLV16, n_traj=n,
                              tspan=(0.0, 6.0), dt=0.1, abstol=1e-6, reltol=1e-6, lanes=ln,
                              maxiters=500, **kw)
        b = runtime.EnsembleBuffers(d, 16, u0, r, A, tspan)
        ctx.solve(d, b, allow=ALLOW)
        out.append(b)
        lanes.append(ctx.stats()["lanes"])
    fields = FIELDS + (("u_saveat",) if kw.get("saveat") is not None else ())
    for f in fields:
        assert bits_equal(out[0].numpy(f), out[1].numpy(f)), f
    return lanes, out[0]


@pytest.mark.parametrize("points,layout,prec", [
    (0, _abi.SAVE_POINT_MAJOR, _abi.PREC_PLAIN), (0, _abi.SAVE_POINT_MAJOR, _abi.PREC_KAHAN),
    (9, _abi.SAVE_POINT_MAJOR, _abi.PREC_PLAIN), (9, _abi.SAVE_TRAJ_MAJOR, _abi.PREC_PLAIN),
    (300, _abi.SAVE_TRAJ_MAJOR, _abi.PREC_PLAIN)])
@pytest.mark.parametrize("n", [65, 129, 1000])
def test_matrix_core_default_has_the_one_lane_bits(ctx, n, points, layout, prec):
    u0, r, A = problem(_abi.RHS_GLV16, n, seed=n)
    ts = np.zeros((2, n))
    ts[1] = np.linspace(0.0, 6.0, n)
    kw = dict(precision=prec, save_layout=layout)
    if points:
        kw["saveat"] = np.linspace(0.0, 6.0, points)
    lanes, _ = _pair(ctx, u0, r, A, ts, **kw)
    assert lanes == [1, 4]


@pytest.mark.parametrize("scale", [1e-45, 1e-40, 1e-38, 1e-30, 1e6, 1e19, 1e30, np.inf, np.nan])
@pytest.mark.parametrize("rate", [0.0, 1e-42, 1.0])
def test_extreme_magnitudes(ctx, scale, rate):
    n = 80
    u0, r, A = problem(_abi.RHS_GLV16, n, seed=3)
    rng = np.random.default_rng(5)
    mix = rng.uniform(size=u0.shape) < 0.4  # some components of each state
    with np.errstate(over="ignore", invalid="ignore"):
        u0 = np.where(mix, u0 * scale, u0).astype(np.float32).astype(np.float64)
    lanes, _ = _pair(ctx, u0, r * rate, A)
    assert lanes == [1, 4]


@pytest.mark.parametrize("kw", [dict(schedule=_abi.SCHED_STAGED), dict(per_lane=1),
                                dict(alg=_abi.ALG_TSIT5)])
def test_one_lane_requests_stay(ctx, kw):
    n = 200
    u0, r, A = problem(_abi.RHS_GLV16, n, seed=4)
    alg = kw.pop("alg", _abi.ALG_ATSIT5)
    d = runtime.make_desc(alg, dtype=_abi.F32, rhs=_abi.RHS_GLV16, n_traj=n, tspan=(0.0, 1.0),
                          dt=0.1, **kw)
    ctx.solve(d, runtime.EnsembleBuffers(d, 16, u0, r, A))
    assert ctx.stats()["lanes"] == 1
