"""Long series (more points than the kernels keep on chip): the fixed-step solvers, whose lanes
are at the same point and load the later times once for all of them, in both precisions and
layouts and at sizes off a wave; and adaptive solves whose lanes stand on both sides of the last
time on chip at once.  Bit for bit against the CPU oracle."""
import numpy as np
import pytest

from helpers import assert_bit_identical, problem, run_pair
from simplediffeq_hip import _abi, runtime

pytestmark = pytest.mark.gpu

FIELDS = ("u_end", "t_end", "retcode", "naccept", "nreject", "u_saveat")


@pytest.mark.parametrize("alg", [_abi.ALG_TSIT5, _abi.ALG_VERN7, _abi.ALG_VERN9])
@pytest.mark.parametrize("n,points,layout", [
    (1, 258, _abi.SAVE_TRAJ_MAJOR), (63, 513, _abi.SAVE_POINT_MAJOR),
    (65, 1025, _abi.SAVE_TRAJ_MAJOR), (300, 2000, _abi.SAVE_POINT_MAJOR)])
def test_fixed_step_series(ctx, alg, n, points, layout):
    u0, p, ps = problem(_abi.RHS_LORENZ, n, seed=points)
    # the last points lie beyond the grid's end and stay unreached
    d = runtime.make_desc(alg, rhs=_abi.RHS_LORENZ, n_traj=n, tspan=(0.0, 1.0), dt=0.01,
                          saveat=np.linspace(0.0, 1.1, points), save_layout=layout)
    st_g, g, st_c, c = run_pair(ctx, d, u0, p, ps)
    assert st_g == st_c == 0
    assert_bit_identical(g, c, FIELDS)


def test_fixed_step_binary32_series_equals_its_short_ones(ctx):
    """binary32 saved points do not depend on how many are asked for."""
    n, points = 130, 600
    u0, p, _ = problem(_abi.RHS_LORENZ, n, seed=4)
    times = np.linspace(0.0, 1.0, points)
    out = []
    for lo, hi in ((0, points), (0, 200), (200, 400), (400, points)):
        d = runtime.make_desc(_abi.ALG_TSIT5, dtype=_abi.F32, n_traj=n, tspan=(0.0, 1.0), dt=0.01,
                              saveat=times[lo:hi])
        b = runtime.EnsembleBuffers(d, 3, u0, p)
        ctx.solve(d, b)
        out.append(b.u_saveat)
    assert np.array_equal(out[0].view(np.int32), np.concatenate(out[1:]).view(np.int32))


@pytest.mark.parametrize("alg", [_abi.ALG_ATSIT5, _abi.ALG_AVERN7])
def test_lanes_on_both_sides_of_the_last_time_on_chip(ctx, alg):
    n, points = 200, 600
    u0, p, ps = problem(_abi.RHS_LORENZ, n, seed=2)
    ts = np.zeros((2, n))
    ts[0] = np.linspace(-1.0, 1.5, n)  # the lanes start up to 300 points apart
    ts[1] = 3.0
    d = runtime.make_desc(alg, rhs=_abi.RHS_LORENZ, n_traj=n, tspan=(0.0, 3.0), dt=0.1,
                          abstol=1e-6, reltol=1e-6, saveat=np.linspace(-1.0, 3.0, points),
                          save_layout=_abi.SAVE_TRAJ_MAJOR)
    st_g, g, st_c, c = run_pair(ctx, d, u0, p, ps, tspan=ts)
    assert st_g == st_c == 0
    assert_bit_identical(g, c, FIELDS)
