"""Binary64 adaptive solves of a wave or two per SIMD run a kernel of their own: around its
sizes' ends, with spans of every length and trajectories that end at once, for every adaptive
solver and small built-in state, the persistent schedule's results bit for bit."""
import numpy as np
import pytest

from helpers import bits_equal
from simplediffeq_hip import _abi, runtime

pytestmark = pytest.mark.gpu

RHS = {1: (_abi.RHS_AFFINE1, 2), 2: (_abi.RHS_LINEAR2, 4), 3: (_abi.RHS_LORENZ, 3)}
SIMD = 4 * 256 * 64  # trajectories of one wave per SIMD


@pytest.mark.parametrize("points", [0, 5, -1])  # -1: every step, packed rows
@pytest.mark.parametrize("alg", [_abi.ALG_ATSIT5, _abi.ALG_AVERN7, _abi.ALG_AVERN9])
@pytest.mark.parametrize("n_state,n", [(3, 1), (3, 63), (3, 65), (1, 1000), (2, 1000), (3, SIMD),
                                       (3, SIMD + 1), (3, 2 * SIMD), (3, 2 * SIMD + 1)])
def test_small_ensembles_have_the_same_bits(ctx, alg, n_state, n, points):
    rhs, n_param = RHS[n_state]
    rng = np.random.default_rng(n)
    u0 = rng.uniform(-1.0, 1.0, (n_state, n))
    p = rng.uniform(0.5, 3.0, (n_param, n))
    ts = np.zeros((2, n))
    ts[1] = rng.uniform(0.0, 3.0, n)
    ts[1, ::7] = 0.0  # an empty span
    dt0 = rng.uniform(1e-6, 0.3, n)
    if n > 10:
        u0[0, 3], dt0[5] = np.inf, 1e-16  # an end by NaN, one by the least step
    out = []
    for sched in (_abi.SCHED_PERSISTENT, _abi.SCHED_AUTO):
        d = runtime.make_desc(alg, rhs=rhs, n_traj=n, dt=0.1, abstol=1e-9, reltol=1e-7,
                              schedule=sched, maxiters=60,
                              saveat=np.linspace(0.0, 3.0, points) if points > 0 else None,
                              save_everystep=points < 0, save_layout=_abi.SAVE_PACKED
                              if points < 0 else _abi.SAVE_POINT_MAJOR)
        b = runtime.EnsembleBuffers(d, n_state, u0, p, tspan=ts, dt0=dt0,
                                    steps_capacity=61 * n if points < 0 else 0)
        ctx.solve(d, b, allow=(_abi.E_DTMIN,))
        out.append(b)
    for f in ("u_end", "t_end", "retcode", "naccept", "nreject") + (("u_saveat",) if points > 0 else ()):
        assert bits_equal(out[0].numpy(f), out[1].numpy(f)), f
    if points < 0:
        rows = int(out[0].steps_offset[n])
        assert bits_equal(out[0].steps_offset, out[1].steps_offset)
        assert bits_equal(out[0].u_steps[:rows], out[1].u_steps[:rows])
        assert bits_equal(out[0].t_steps[:rows], out[1].t_steps[:rows])
