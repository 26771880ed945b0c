"""Save times kept on chip (the first 256) and those beyond them: ensembles that save one
point fewer, as many, one more and many more than that, in every lane layout and the
fixed-step solvers, bit for bit against the CPU oracle."""
import numpy as np
import pytest

from helpers import assert_bit_identical, problem, run_pair
from simplediffeq_hip import _abi, runtime

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("points", [1, 255, 256, 257, 700])
@pytest.mark.parametrize("rhs,alg,lanes,dtype", [
    (_abi.RHS_LORENZ, _abi.ALG_ATSIT5, 1, _abi.F64), (_abi.RHS_LORENZ, _abi.ALG_AVERN7, 1, _abi.F64),
    (_abi.RHS_GLV16, _abi.ALG_AVERN9, 4, _abi.F64), (_abi.RHS_GLV16, _abi.ALG_ATSIT5, 16, _abi.F64),
    (_abi.RHS_LORENZ, _abi.ALG_TSIT5, 1, _abi.F64), (_abi.RHS_LORENZ, _abi.ALG_VERN9, 1, _abi.F64)])
def test_save_times(ctx, rhs, alg, lanes, dtype, points):
    n = 67
    u0, p, ps = problem(rhs, n, seed=points)
    adaptive = alg in (_abi.ALG_ATSIT5, _abi.ALG_AVERN7, _abi.ALG_AVERN9)
    d = runtime.make_desc(alg, dtype=dtype, rhs=rhs, n_traj=n, tspan=(0.0, 3.0),
                          dt=0.1 if adaptive else 0.01, abstol=1e-6, reltol=1e-6, lanes=lanes,
                          saveat=np.linspace(0.0, 3.0, points), save_layout=_abi.SAVE_TRAJ_MAJOR)
    st_g, g, st_c, c = run_pair(ctx, d, u0, p, ps)
    assert st_g == st_c == 0
    assert_bit_identical(g, c, ("u_end", "t_end", "retcode", "naccept", "nreject", "u_saveat"))
