"""The controller's logarithm and power for an error estimate in its checked range
(log_in_dd, pow_in): the bits of the general pow_log / pow_from_ctrl, on the device, over
the whole range of estimates [2^-351, 2^350] and its ends."""
import numpy as np
import pytest

from helpers import bits_equal
from simplediffeq_hip import _abi, runtime

pytestmark = pytest.mark.gpu

SRC = """
template <class T>
__device__ void probe(T* du, const T* u, const T* p, const T* __restrict__ ps, double t) {
  const sdeh_math::ConstTab tab;
  double hi, lo;
  sdeh_math::log_in_dd(p[0], &hi, &lo, tab);
  const sdeh_math::PowLog l = sdeh_math::pow_log_ctrl(p[0], tab);
  du[0] = sdeh_math::pow_in(hi, lo, p[1], tab);
  du[1] = sdeh_math::pow_from_ctrl(l, p[1], tab);
  du[2] = sdeh::Ops<double>::max_abs(p[0], -p[1]);
  du[3] = sdeh::Ops<double>::min_abs(-p[0], p[1]);
}
"""


@pytest.mark.parametrize("beta", [0.7 / 5, 0.4 / 5, 0.7 / 7, 0.4 / 7, 0.7 / 9, 0.4 / 9])
def test_in_range_power_is_the_general_power(ctx, beta):
    rng = np.random.default_rng(int(beta * 1e6))
    n = 20000
    x = np.ldexp(rng.uniform(1.0, 2.0, size=n), rng.integers(-351, 350, size=n))
    near = np.ldexp(rng.uniform(0.5, 2.0, size=n // 2), rng.integers(-8, 4, size=n // 2))
    x[: n // 2] = near
    one = 1.0
    x[:8] = [2.0 ** -351, 2.0 ** 350, one, np.nextafter(one, 0), np.nextafter(one, 2), 1e-4,
             np.nextafter(2.0 ** 350, 0), 0.69]
    h = ctx.compile_rhs(SRC, "probe", 4, 2)
    d = runtime.make_desc(_abi.ALG_EULER, rhs=h, n_traj=n, tspan=(0.0, 1.0), dt=1.0)
    buf = runtime.EnsembleBuffers(d, 4, np.zeros((4, n)), np.stack([x, np.full(n, beta)]))
    assert ctx.solve(d, buf) == 0
    got = buf.u_end
    assert bits_equal(got[0], got[1])
    assert bits_equal(got[2], np.maximum(x, beta))
    assert bits_equal(got[3], np.minimum(x, beta))
