"""A registered right-hand side whose sector-writing kernel does not compile: the ranked saving
pass writes row by row instead, with the same rows, leaves no error message behind a call that
succeeded, and does not compile again on the next one."""
import time

import numpy as np
import pytest

from helpers import bits_equal
from simplediffeq_hip import _abi, runtime

pytestmark = pytest.mark.gpu

# the specialization makes the library's own check on the state's size refuse that kernel alone
NO_SECTORS = """
struct sdeh_user_rhs;
namespace sdeh {
template <> struct PkWave<double, sdeh_user_rhs> { static constexpr bool value = false; };
}
"""
DECAY = """
template <class T> __device__ inline void %s(T* du, const T* u, const T* p, const T* ps, double t) {
  du[0] = p[0] * u[1];
  du[1] = -p[0] * u[0];
}
"""


def test_row_by_row_where_the_sector_kernel_is_missing():
    c = runtime.Context(0)
    n = 400_001  # beyond what fits the GPU at once
    rng = np.random.default_rng(3)
    u0, p = rng.uniform(-1.0, 1.0, (2, n)), rng.uniform(0.5, 3.0, (1, n))
    out = []
    for head, name in (("", "turn_a"), (NO_SECTORS, "turn_b")):
        rhs = c.compile_rhs(head + DECAY % name, name, 2, 1)
        d = runtime.make_desc(_abi.ALG_ATSIT5, rhs=rhs, n_traj=n, tspan=(0.0, 0.5), dt=0.1,
                              abstol=1e-6, reltol=1e-5, save_everystep=True,
                              save_layout=_abi.SAVE_PACKED)
        b = runtime.EnsembleBuffers(d, 2, u0, p, backend="torch", device="cuda:0",
                                    steps_capacity=20 * n)
        b.u_steps.fill_(-5.5)
        b.t_steps.fill_(-5.5)
        took = []
        for _ in range(2):
            t0 = time.perf_counter()
            assert c.solve(d, b) == 0
            took.append(time.perf_counter() - t0)
            assert c.last_error() == ""
        assert c.stats()["schedule"] == _abi.SCHED_ONE_LAUNCH
        assert took[1] < 0.5 * took[0]  # the first call compiles
        out.append(b)
    for f in ("u_end", "t_end", "naccept", "n_steps", "steps_offset", "u_steps", "t_steps"):
        assert bits_equal(out[0].numpy(f), out[1].numpy(f)), f
    c.close()
